// Products of any number of tokens: y[N, M] = x[N, K] @ dequant(W[M, K])^T, token-major on both
// sides (K fastest in x, M fastest in y), so callers transpose nothing.  The windows of 32 and 64
// columns (nf4_gemm.hip) read and decode the whole matrix once per window; here a workgroup keeps
// 256 or 512 weight rows against up to 128 tokens, so a matrix is decoded once per 128 tokens.
// Bound: up to about 64 tokens the bytes of the weights and a workgroup's fixed start, above the
// matrix cores and the LDS reads beside them.  Whole calls through the linear seat from a graph, windows
// of 32 before and this after (us): 512x512 at 8 tokens 11.2 / 8.0, 5120x5120 at 17 27.4 / 14.9 and at
// 32 19.2 / 16.7, 13824x5120 at 64 47 / 33, 11008x2048 at 333 189 / 43, 5120x13824 at 1024 797 / 167 (870
// TFLOP/s; the library's dense bf16 8192^3 product reaches 1150 on this card).  A window of whole vectors
// is still the faster through some matrices of 10^8 codes and more: 16384x6144 at 8 / 32 tokens 24.7 / 27.7
// and 25.9 / 29.5, 27648x5184 at 8 37.5 and 42.4, a ragged 16384x6100 at 32 27.7 and 33.6.
//
// Arithmetic: bf16(kWideUnit * level) times the bf16 activation in the matrix cores, every 64-wide
// group's sum times its scale / kWideUnit in fp32, splits added in fp32 in a fixed order, one bf16
// rounding.

#include "nf4_common.h"

#include <cmath>

namespace chr {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 Bf16x8;
typedef __attribute__((ext_vector_type(4))) float F32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t Raw16;

// The levels as the matrix cores take them.  A level rounded to bf16 is off by the same amount in
// every weight that has it, so what the sixteen errors leave on average grows with the sum of x: with
// bf16(level) a product of activations that do not average to zero (behind a relu or a gate) was off
// by 2e-2 of its norm at K = 5120, 4e-2 at 27648.  The unit and three other roundings were chosen for
// errors that are small (1.13e-3 of the weights' norm; bf16(level) 1.38e-3, bf16(level * scale)
// 1.66e-3) and cancel: levels 1, 6 and 10 are rounded to the nearest in lanes of even 16-lane rows
// and to the neighbour on the other side in odd ones, which take the other half of every group's K.
// The average left is below 3e-6 of the weights' norm, whether they are normal, Laplace, uniform,
// triangular or Student-t (bf16(level) 4e-4).  Products of K = 1024 .. 27648 against 64 bits, x of zero
// mean, of mean 1 and sigma 0.3, and behind a relu or silu: 1.8e-3 .. 2.1e-3 of the norm, the rounding
// of the result (1.7e-3) included.
constexpr float kWideUnit = 1.24227f;
constexpr uint32_t kWideLevel[16] = {0xBF9F, 0xBF5D, 0xBF27, 0xBEFB, 0xBEB5, 0xBE6B, 0xBDE8, 0x0000,
                                     0x3DCA, 0x3E4D, 0x3E9D, 0x3ED7, 0x3F0C, 0x3F33, 0x3F66, 0x3F9F};
constexpr int kWideOther[16] = {0, 1, 0, 0, 0, 0, -1, 0, 0, 0, -1};  // to the neighbour in odd 16-lane rows

struct WideArgs {
  const uint8_t *packed;
  const uint16_t *scale;
  const uint16_t *x;
  uint16_t *y;
  float *part;  // fp32 partials [splits][N][M], or null
  const uint16_t *bias;
  int64_t x_stride;
  int N, M, K;
  int groups, split_groups;
  int tiles_m, tiles_n;
};

// A wavefront owns 64 weight rows and TT * 16 tokens; WM x WN wavefronts make the tile.
//
// Weights never pass through LDS: the tokens are the rows of the MFMA's result and the weight rows
// its columns, so lane l holds column l % 16 and the scale of a row is a register of the lanes
// that hold its column.  The 16-row block t takes rows 4i + t (i = l % 16): a lane ends with four
// consecutive features of each of its tokens and stores them as one 8-byte vector.  A row's 16-byte
// load covers two groups from four lanes 16 apart; one half-wavefront swap per dword pair
// (v_permlane32_swap) leaves each group spread over all four, codes {0, 32, 16, 48}[l / 16] ..+15
// of it, and x is read from LDS in the same order.  The loads themselves go by the row's lines: four
// neighbouring lanes take a row's 64 bytes and a ds_bpermute hands the pieces over, and a lane
// fetches the scales of one row for the whole wavefront through LDS (with every lane loading its own
// four rows' pieces and scales 5120x5120 at 512 tokens unsplit took 325 us, so 161).  Bytes become
// bf16 pairs through the per-lane table of nf4_common.h (64 KB, one address op and one conflict-free
// read per two weights); 128 tokens a wavefront halve the lookups per product against 64.
//
// x goes from global memory straight to LDS one stage of two groups ahead, 128-byte rows whose 16-byte
// pieces are XORed with the row's low bits: the 16-lane reads of a fragment touch all banks once.
//
// WHOLE: the rows of x are whole 16-byte pieces of whole groups.  Otherwise (a ragged K, rows at any
// 2-byte boundary) the pieces pass through registers, what lies behind K as zeros: a padded copy is two
// launches (at 8 tokens 320x500 17.1 us, 12.7 so; 16384x6100 34.8, 29.3, each with a slower table fill), but the 512 x 128 tile spills
// five registers and runs a tenth longer, so large calls bring one (16384x6100 at 1024 tokens 215 us,
// 235 so).
template <int WM, int WN, int TT, bool WHOLE>
__global__ __launch_bounds__(WM *WN *kWave) void wide_gemm(const WideArgs a) {
  constexpr int NW = WM * WN;
  constexpr int BN = WN * TT * 16;
  constexpr int kStageBytes = 2 * BN * 128;  // two groups of 64 K
  constexpr int kBlocks = 2 * BN / 8;  // 1 KB pieces of a stage, one per wavefront and pass
  static_assert(kBlocks % NW == 0, "stage pieces must divide over the wavefronts");
  constexpr int kPass = kBlocks / NW;
  extern __shared__ __align__(16) uint32_t smem[];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int wm = wave / WN, wn = wave % WN;
  const int li = lane & 15, lg = lane >> 4;
  const uint32_t lane4 = static_cast<uint32_t>(lane) * 4;

  // Workgroups are dealt to the eight XCDs in turn: each XCD takes a contiguous run of tiles,
  // token tiles fastest, so the tiles that share weight rows meet in one L2.
  const int total = static_cast<int>(gridDim.x);
  const int xcd = static_cast<int>(blockIdx.x) & 7;
  const int per = total >> 3, rem = total & 7;
  const int tile = xcd * per + min(xcd, rem) + (static_cast<int>(blockIdx.x) >> 3);
  const int tn = tile % a.tiles_n;
  const int tms = tile / a.tiles_n;
  const int tm = tms % a.tiles_m;
  const int split = tms / a.tiles_m;
  const int g_lo = split * a.split_groups;
  const int g_hi = min(g_lo + a.split_groups, a.groups);

  // The four weight rows whose codes this lane fetches (16 bytes of each: four lanes take a row's 64),
  // as two pairs of neighbours, and the one row whose scales it fetches; rows past the end are
  // clamped, computed and not stored.
  const int m0 = (tm * WM + wm) * 64;
  const int row_bytes = a.groups * 32;
  const uint8_t *wp[2];
  int wd[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int want = m0 + 4 * (lane >> 2) + 2 * h;
    wp[h] = a.packed + static_cast<size_t>(min(want, a.M - 1)) * row_bytes + (lane & 3) * 16;
    wd[h] = want + 1 < a.M ? row_bytes : 0;
  }
  const int from_lane4 = (4 * li + lg) * 4;
  const uint16_t *sp = a.scale + static_cast<size_t>(min(m0 + lane, a.M - 1)) * a.groups;

  const int tok0 = tn * BN;
  const uint16_t *xp[kPass];
#pragma unroll
  for (int p = 0; p < kPass; ++p) {
    const int b = wave + p * NW;
    const int sub = b / (BN / 8);
    const int row = (b % (BN / 8)) * 8 + (lane >> 3);
    const int piece = (lane & 7) ^ (lane >> 3);
    xp[p] = a.x + static_cast<int64_t>(min(tok0 + row, a.N - 1)) * a.x_stride + sub * kGroup + piece * 8;
  }

  uint4 xr[WHOLE ? 1 : kPass];
  auto load_x = [&](int g, int buf) {
#pragma unroll
    for (int p = 0; p < kPass; ++p) {
      // the second half of a last, odd stage is not multiplied: it reads its first half again
      const int sub = (wave + p * NW) / (BN / 8);
      const int off = (sub == 1 && g + 1 >= g_hi) ? (g - 1) * kGroup : g * kGroup;
      if constexpr (WHOLE) {
        const uint32_t at = static_cast<uint32_t>(kPairTableBytes + buf * kStageBytes + (wave + p * NW) * 1024);
        load_to_lds16(xp[p] + off, at);
      } else if ((g + 2) * kGroup <= a.K) {
        __builtin_memcpy(&xr[p], xp[p] + off, 16);
      } else {
        const int left = a.K - off - sub * kGroup - ((lane & 7) ^ (lane >> 3)) * 8;
        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (e < left) {
            w[e >> 1] |= static_cast<uint32_t>(xp[p][off + e]) << (16 * (e & 1));
          }
        }
        xr[p] = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
  };
  auto store_x = [&](int buf) {
    if constexpr (!WHOLE) {
#pragma unroll
      for (int p = 0; p < kPass; ++p) {
        const uint32_t at = static_cast<uint32_t>(kPairTableBytes + buf * kStageBytes + (wave + p * NW) * 1024 + lane * 16);
        *reinterpret_cast<__attribute__((address_space(3))) Raw16 *>(at) = __builtin_bit_cast(Raw16, xr[p]);
      }
    }
  };
  auto from_loader = [&](uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from_lane4, static_cast<int>(v)));
  };
  uint4 cw[4], nw[4];
  uint32_t ns01;
  // codes and scales of groups g and g + 1 (a last odd group: its own twice)
  auto load_w = [&](int g, uint4 (&w)[4]) {
    const bool odd = g + 1 >= g_hi;
    const int at = g * 32 - (odd && (lane & 2) != 0 ? 32 : 0);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      w[t] = *reinterpret_cast<const uint4 *>(wp[t >> 1] + at + ((t & 1) != 0 ? wd[t >> 1] : 0));
    }
    // both scales in one load, at whatever 2-byte boundary the row puts them: each of its 64 lanes
    // reads a line of its own, and as two loads an odd group count cost a third more than its even
    // neighbour (16 tokens, 16384x6208 42.6 us against 30.8 at 6272; 29.8 and 28.4 so)
    if (odd) {
      ns01 = sp[g];
    } else {
      __builtin_memcpy(&ns01, sp + g, 4);
    }
  };
  // a wavefront's scales of two groups, by row: lane i reads the four of its rows 4i .. 4i + 3
  const uint32_t sc_at = static_cast<uint32_t>(kPairTableBytes + 2 * kStageBytes + wave * 512);
  auto store_s = [&]() {
    *reinterpret_cast<__attribute__((address_space(3))) float *>(sc_at + lane * 4) = f16_to_f32(static_cast<uint16_t>(ns01)) * (1.f / kWideUnit);
    *reinterpret_cast<__attribute__((address_space(3))) float *>(sc_at + 256 + lane * 4) = f16_to_f32(static_cast<uint16_t>(ns01 >> 16)) * (1.f / kWideUnit);
  };
  auto read_s = [&](int half) {
    return __builtin_bit_cast(F32x4, lds0_u128(sc_at + half * 256 + li * 16));
  };

  load_x(g_lo, 0);
  load_w(g_lo, cw);
  // The table, sixteen bytes of one high code at a time, their low levels literals: an instruction and
  // half a store a byte.  One byte a turn, its two levels loaded, took 4 us of every workgroup's start (from
  // a graph 512x512 at 8 tokens 12.0 us, 8.0 so; 5120x5120 at 17 18.1 and 14.9).
  const uint32_t odd_row = (lane >> 4) & 1;
  uint32_t hi[16 / NW];
#pragma unroll
  for (int i = 0; i < 16 / NW; ++i) {
    hi[i] = (kWideLevel[wave + i * NW] + static_cast<uint32_t>(kWideOther[wave + i * NW]) * odd_row) << 16;
  }
#pragma unroll
  for (int i = 0; i < 16 / NW; ++i) {
#pragma unroll
    for (int l = 0; l < 16; ++l) {
      smem[(16 * (wave + i * NW) + l) * 64 + lane] =
          hi[i] | (kWideLevel[l] + static_cast<uint32_t>(kWideOther[l]) * odd_row);
    }
  }
  store_s();
  store_x(0);
  lds_loads_done();
  __syncthreads();

  F32x4 acc[TT][4];
#pragma unroll
  for (int i = 0; i < TT; ++i) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc[i][t] = F32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  const uint32_t piece0 = static_cast<uint32_t>((((lg & 1) << 2) | (lg & 2)) ^ (li & 7));

  // one group: `lo`/`hi` are the lane's 16 codes of each of its rows
  auto group = [&](uint32_t xbase, const uint32_t (&lo)[4], const uint32_t (&hi)[4], const F32x4 s) {
    Bf16x8 wf[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const Raw16 r0 = {pair_at<0>(lo[t], lane4), pair_at<1>(lo[t], lane4), pair_at<2>(lo[t], lane4), pair_at<3>(lo[t], lane4)};
      const Raw16 r1 = {pair_at<0>(hi[t], lane4), pair_at<1>(hi[t], lane4), pair_at<2>(hi[t], lane4), pair_at<3>(hi[t], lane4)};
      wf[t][0] = __builtin_bit_cast(Bf16x8, r0);
      wf[t][1] = __builtin_bit_cast(Bf16x8, r1);
    }
    const uint32_t row0 = xbase + static_cast<uint32_t>((wn * TT * 16 + li) * 128);
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      const uint32_t at = row0 + static_cast<uint32_t>(i * 16 * 128);
      const Bf16x8 x0 = __builtin_bit_cast(Bf16x8, lds0_u128(at + piece0 * 16));
      const Bf16x8 x1 = __builtin_bit_cast(Bf16x8, lds0_u128(at + (piece0 ^ 1) * 16));
      F32x4 d[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0, wf[t][0], F32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x1, wf[t][1], d[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[i][t][r] = fmaf(d[t][r], s[t], acc[i][t][r]);
        }
      }
    }
  };

  int buf = 0;
  for (int g = g_lo; g < g_hi; g += 2) {
    const bool two = g + 1 < g_hi;
    const bool more = g + 2 < g_hi;
    const uint32_t base0 = static_cast<uint32_t>(kPairTableBytes + buf * kStageBytes);
    if (more) {
      load_x(g + 2, buf ^ 1);
    }
    uint32_t lo[4], hi[4], lo2[4], hi2[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const auto p0 = __builtin_amdgcn_permlane32_swap(from_loader(cw[t].x), from_loader(cw[t].z), false, false);
      const auto p1 = __builtin_amdgcn_permlane32_swap(from_loader(cw[t].y), from_loader(cw[t].w), false, false);
      lo[t] = p0[0];
      hi[t] = p1[0];
      lo2[t] = p0[1];
      hi2[t] = p1[1];
    }
    if (more) {
      load_w(g + 2, nw);
    }
    const F32x4 s0 = read_s(0), s1 = read_s(1);
    group(base0, lo, hi, s0);
    if (two) {
      group(base0 + BN * 128, lo2, hi2, s1);
    }
    if (more) {
      store_s();
      store_x(buf ^ 1);
    }
    lds_loads_done();
    __syncthreads();
    buf ^= 1;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      cw[t] = nw[t];
    }
  }

  const int tok_w = tok0 + wn * TT * 16 + lg * 4;
  const int m = m0 + 4 * li;
  if (a.part != nullptr) {
    float *part = a.part + static_cast<size_t>(split) * a.N * a.M;
#pragma unroll
    for (int i = 0; i < TT; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = tok_w + i * 16 + r;
        if (tok >= a.N) {
          continue;
        }
        float *dst = part + static_cast<size_t>(tok) * a.M + m;
        if ((a.M & 3) == 0) {
          if (m < a.M) {
            *reinterpret_cast<F32x4 *>(dst) = F32x4{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
          }
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            if (m + t < a.M) {
              dst[t] = acc[i][t][r];
            }
          }
        }
      }
    }
    return;
  }
  float b[4] = {0.f, 0.f, 0.f, 0.f};
  if (a.bias != nullptr) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      b[t] = bf16_to_f32(a.bias[min(m + t, a.M - 1)]);
    }
  }
#pragma unroll
  for (int i = 0; i < TT; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = tok_w + i * 16 + r;
      if (tok >= a.N) {
        continue;
      }
      uint16_t o[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        o[t] = f32_to_bf16(acc[i][t][r]);
        if (a.bias != nullptr) {
          o[t] = f32_to_bf16(bf16_to_f32(o[t]) + b[t]);
        }
      }
      uint16_t *dst = a.y + static_cast<size_t>(tok) * a.M + m;
      if ((a.M & 3) == 0) {
        if (m < a.M) {
          *reinterpret_cast<uint2 *>(dst) = make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16),
                                                       o[2] | (static_cast<uint32_t>(o[3]) << 16));
        }
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (m + t < a.M) {
            dst[t] = o[t];
          }
        }
      }
    }
  }
}

// W partials of one row added over the splits, in split order.
template <int W>
__device__ __forceinline__ void sum_splits(const float *p, int splits, int64_t stride, float (&v)[W]) {
#pragma unroll
  for (int e = 0; e < W; ++e) {
    v[e] = 0.f;
  }
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    if constexpr (W == 4) {
      const F32x4 t = *reinterpret_cast<const F32x4 *>(p + s * stride);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] += t[e];
      }
    } else {
      v[0] += p[s * stride];
    }
  }
}

template <int W>
__device__ __forceinline__ void store_bf16(uint16_t *dst, const uint16_t (&o)[W]) {
  if constexpr (W == 4) {
    *reinterpret_cast<uint2 *>(dst) =
        make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16), o[2] | (static_cast<uint32_t>(o[3]) << 16));
  } else {
    dst[0] = o[0];
  }
}

// y = bf16(sum of the splits) (+ bias), W features a thread.
template <int W>
__global__ __launch_bounds__(256) void wide_reduce(const float *__restrict__ part, int splits, int64_t count, int M,
                                                   const uint16_t *__restrict__ bias, uint16_t *__restrict__ y) {
  const int64_t at = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * W;
  if (at >= count) {
    return;
  }
  const int m = static_cast<int>(at % M);
  uint16_t o[W];
  float v[W];
  sum_splits<W>(part + at, splits, count, v);
#pragma unroll
  for (int e = 0; e < W; ++e) {
    o[e] = f32_to_bf16(v[e]);
    if (bias != nullptr) {
      o[e] = f32_to_bf16(bf16_to_f32(o[e]) + bf16_to_f32(bias[m + e]));
    }
  }
  store_bf16<W>(y + at, o);
}

template <int WM, int WN, int TT, bool WHOLE>
int wide_launch(WideArgs &a, int splits, hipStream_t st) {
  constexpr int BN = WN * TT * 16;
  constexpr int kLds = kPairTableBytes + 4 * BN * 128 + WM * WN * 512;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(&wide_gemm<WM, WN, TT, WHOLE>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess) {
    (void)hipGetLastError();
    return -6;
  }
  const int bm = WM * 64;
  a.tiles_m = (a.M + bm - 1) / bm;
  a.tiles_n = (a.N + BN - 1) / BN;
  const int64_t grid = static_cast<int64_t>(a.tiles_m) * a.tiles_n * splits;
  if (grid > INT32_MAX) {
    return -3;
  }
  wide_gemm<WM, WN, TT, WHOLE><<<dim3(static_cast<unsigned>(grid)), dim3(WM * WN * kWave), kLds, st>>>(a);
  return launch_rc();
}

// ---- tile and split choice -------------------------------------------------------------------
// A compute unit holds one workgroup (64 KB of table).  The cost in us, fitted to an MI355X: a round
// of workgroups takes a fixed part (launch, table, first loads, stores) and a part per group of 64 K,
// splits add 3.5 and the writing and reading of their fp32 partials at 3.4 TB/s together.  Unsplit
// 8 / 32 / 80 / 216 groups took 11 / 26 / 54 / 132 us on 256 x 16, 17 / 42 / 92 / 230 on 256 x 64 and
// 18 / 48 / 111 / 285 on 256 x 128; 80 groups 161 on 512 x 128, which does the most a us where it fills
// the chip.  (All with a table fill that took 4 us longer.  The fixed parts stand as they were: taken off,
// they send 512x512 at 8 tokens to splits and a second launch, 6.3 us from a graph instead of 8.0 but 19.8
// instead of 15.8 in a program that calls it launch by launch, and change no larger call by more than 3%.)
// At 5120 x 5120, then: 17 tokens 17.7 us on 256 x 32 in 10 splits (23.8 on 256 x 64), 128 tokens
// 32 us on 256 x 64 in 6 (44 on 512 x 128), 512 tokens 57 on 512 x 128 in 6 (100 on 256 x 64).
struct WideTile {
  int wm, bn;
  float fixed, per_group;
};
constexpr WideTile kWideTiles[] = {
    {8, 128, 9.f, 1.9f}, {4, 128, 7.5f, 1.28f}, {4, 64, 9.f, 1.03f}, {4, 32, 7.6f, 0.71f}, {4, 16, 7.f, 0.58f}};
constexpr int kWideMaxSplits = 32;

struct WidePlan {
  int tile, splits, split_groups;
};

WidePlan wide_plan(int M, int N, int groups) {
  WidePlan best{0, 1, groups};
  float best_us = 3.0e38f;
  const float cus = static_cast<float>(device_cu_count());
  for (int t = 0; t < static_cast<int>(sizeof(kWideTiles) / sizeof(kWideTiles[0])); ++t) {
    const WideTile &w = kWideTiles[t];
    const float tiles = static_cast<float>((M + w.wm * 64 - 1) / (w.wm * 64)) * static_cast<float>((N + w.bn - 1) / w.bn);
    for (int want = 1; want <= kWideMaxSplits; ++want) {
      const int per = ((groups + want - 1) / want + 1) / 2 * 2;  // whole stages of two groups
      const int splits = (groups + per - 1) / per;
      if (splits != want) {
        continue;
      }
      float us = ceilf(tiles * static_cast<float>(splits) / cus) *
                 (w.fixed + w.per_group * static_cast<float>(per < groups ? per : groups));
      if (splits > 1) {
        us += 3.5f + 4.f * static_cast<float>(splits) * static_cast<float>(N) * static_cast<float>(M) / 3.4e6f;
      }
      if (us < best_us) {
        best_us = us;
        best = WidePlan{t, splits, per};
      }
    }
  }
  return best;
}

template <bool WHOLE>
int wide_dispatch(int tile, WideArgs &a, int splits, hipStream_t st) {
  switch (tile) {
    case 0: return wide_launch<8, 1, 8, WHOLE>(a, splits, st);
    case 1: return wide_launch<4, 2, 4, WHOLE>(a, splits, st);
    case 2: return wide_launch<4, 1, 4, WHOLE>(a, splits, st);
    case 3: return wide_launch<4, 1, 2, WHOLE>(a, splits, st);
    default: return wide_launch<4, 1, 1, WHOLE>(a, splits, st);
  }
}

// Descriptor checks and the launch arguments the matrix decides.
int wide_args(const chr_nf4_dev_t *w, int32_t N, WideArgs &a) {
  if (w == nullptr) {
    return -1;
  }
  if (N < 1) {
    return -2;
  }
  if (w->M < 1 || w->K < 1 || w->packed == nullptr || w->scale == nullptr || w->M > INT32_MAX / 2 ||
      w->K > INT32_MAX / 64) {
    return -3;
  }
  if (!k_pad_ok(w->K, w->K_pad)) {
    return -4;
  }
  if (!aligned16(w->packed) || !aligned2(w->scale)) {
    return -5;
  }
  a.packed = w->packed;
  a.scale = w->scale;
  a.M = w->M;
  a.K = w->K;
  a.N = N;
  a.groups = w->K_pad / kGroup;
  return 0;
}

int64_t wide_ws(const WideArgs &a, const WidePlan &p) {
  return p.splits == 1 ? 0 : static_cast<int64_t>(p.splits) * a.N * a.M;
}

// rows: x at any 2-byte boundary, its rows x_stride >= K apart.  Otherwise whole 16-byte pieces of
// whole groups, a ragged K padded by the caller.
int wide_entry(const chr_nf4_dev_t *w, const void *x, int64_t x_stride, int32_t N, void *y, float *ws, int64_t ws_floats,
               const void *bias, void *stream, bool rows) {
  if (x == nullptr || y == nullptr) {
    return -1;
  }
  WideArgs a{};
  if (const int rc = wide_args(w, N, a)) {
    return rc;
  }
  if (rows ? x_stride < w->K : (x_stride < w->K_pad || (x_stride & 7) != 0)) {
    return -3;
  }
  const WidePlan p = wide_plan(a.M, N, a.groups);
  const int64_t need = wide_ws(a, p);
  if (!(rows ? aligned2(x) : aligned16(x)) || (reinterpret_cast<uintptr_t>(y) & 7u) != 0 || (need > 0 && !aligned16(ws))) {
    return -5;
  }
  if (need > 0 && (ws == nullptr || ws_floats < need)) {
    return -7;
  }
  const bool vec = (a.M & 3) == 0;
  const int64_t count = static_cast<int64_t>(N) * a.M;
  const int64_t blocks = (count / (vec ? 4 : 1) + 255) / 256;
  if (blocks > INT32_MAX) {
    return -3;
  }
  a.x = static_cast<const uint16_t *>(x);
  a.x_stride = x_stride;
  a.y = static_cast<uint16_t *>(y);
  a.bias = static_cast<const uint16_t *>(bias);
  a.part = need > 0 ? ws : nullptr;
  a.split_groups = p.split_groups;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool whole = !rows || (w->K == w->K_pad && (x_stride & 7) == 0 && aligned16(x));
  const int rc = whole ? wide_dispatch<true>(p.tile, a, p.splits, st) : wide_dispatch<false>(p.tile, a, p.splits, st);
  if (rc != 0 || a.part == nullptr) {
    return rc;
  }
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  if (vec) {
    wide_reduce<4><<<grid, block, 0, st>>>(a.part, p.splits, count, a.M, a.bias, a.y);
  } else {
    wide_reduce<1><<<grid, block, 0, st>>>(a.part, p.splits, count, a.M, a.bias, a.y);
  }
  return launch_rc();
}

}  // namespace
}  // namespace chr

using namespace chr;

extern "C" int64_t chr_nf4_wide_ws(const chr_nf4_dev_t *w, int32_t N) {
  WideArgs a{};
  if (wide_args(w, N, a) != 0) {
    return -1;
  }
  return wide_ws(a, wide_plan(a.M, N, a.groups));
}

extern "C" int chr_nf4_wide_plan(const chr_nf4_dev_t *w, int32_t N, int32_t *rows, int32_t *tokens, int32_t *splits) {
  WideArgs a{};
  if (rows == nullptr || tokens == nullptr || splits == nullptr) {
    return -1;
  }
  if (const int rc = wide_args(w, N, a)) {
    return rc;
  }
  const WidePlan p = wide_plan(a.M, N, a.groups);
  *rows = kWideTiles[p.tile].wm * 64;
  *tokens = kWideTiles[p.tile].bn;
  *splits = p.splits;
  return 0;
}

extern "C" int chr_nf4_wide(const chr_nf4_dev_t *w, const void *x, int64_t x_stride, int32_t N, void *y, float *ws,
                            int64_t ws_floats, const void *bias, void *stream) {
  return wide_entry(w, x, x_stride, N, y, ws, ws_floats, bias, stream, false);
}

extern "C" int chr_nf4_wide_rows(const chr_nf4_dev_t *w, const void *x, int64_t x_stride, int32_t N, void *y, float *ws,
                                 int64_t ws_floats, const void *bias, void *stream) {
  return wide_entry(w, x, x_stride, N, y, ws, ws_floats, bias, stream, true);
}
