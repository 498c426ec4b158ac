// Several whole windows of a prompt at once, with the bits of one window after the other.
//
// The chunk prefill (dv2_prefill.hip, gemm_stream64 in nf4_gemm.hip) takes 64 tokens at a time: every
// window reads and decodes all weights again, in launches too short to fill the chip.  Activations of
// 48 to 64 layers in bf16 carry any change of a sum's order into every later element, so these
// kernels keep each sum in the window's order -- the products group by group as the 64-column tile
// adds them, the norms' squares block by block as that tile and rms_cols add them -- and change only
// which launch and workgroup a token is computed in.  All data is token-major, [N, features] with
// N a multiple of 64.

#include "nf4_common.h"

namespace chr {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 Bf16x8;
typedef __attribute__((ext_vector_type(4))) float F32x4;
typedef __attribute__((ext_vector_type(16))) float F32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t Raw16;

constexpr int kPromptMats = 3;
constexpr int kWindow = 64;       // tokens of a window, and of a workgroup here
constexpr int kChunk = 256;       // K of a stage: four groups, as in the 64-column tile
constexpr int kBlocks = 4;        // 32-row blocks of a wavefront
constexpr int kTileRows = 2 * kBlocks * 32;
constexpr int kXStage = kWindow * kChunk * 2;
constexpr int kScaleStage = 4 * kTileRows * 2;
constexpr int kXAddr = kPairTableBytes;
constexpr int kScaleAddr = kXAddr + 2 * kXStage;
constexpr int kPromptLds = kScaleAddr + 2 * kScaleStage;
constexpr int kPromptThreads = 512;

struct PromptArgs {
  const uint8_t *packed[kPromptMats];
  const uint16_t *scale[kPromptMats];
  int first[kPromptMats + 1];  // concatenated row each matrix starts at
  const uint16_t *x;
  uint16_t *y;
  float *part;  // [splits][N][rows] (SwiGLU: gate features, then up), or null
  const uint16_t *bias;
  int M;        // output features; of one matrix when PAIR
  int N, K, chunks, split_chunks, tiles_m, tiles_n;
};

__device__ __forceinline__ uint16_t swiglu_bf16(float gate, float up) {
  const float a = bf16_to_f32(f32_to_bf16(gate));
  const float act = bf16_to_f32(f32_to_bf16(a / (1.f + expf(-a))));
  return f32_to_bf16(act * bf16_to_f32(f32_to_bf16(up)));
}

// Bound: a chunk of 256 K takes 4050 clocks of which the matrix cores work 2048; the rest is the vector
// instructions that do not fit beside them (a scaling per product and token, an address per two weights), LDS
// and the start of a chunk; 18 000 clocks a workgroup lie outside the loop.  Gate and up of 27648 x 5120 at
// 1792 tokens 1.38 ms (0.74 PFLOP/s; 1.70 with every block's lookups, products and scaling one after the
// other), down 5120 x 27648 0.70 (0.89), at 512 tokens 13824 x 5120 207 us (263), 5120 x 13824 104 (132),
// 5120 x 5120 55 (69), 7168 x 5120 68 (86); on a faster card 1.24 and 0.67 ms, 192, 90, 45 and 57 us.  There the
// matrix cores are busy 0.33 to 0.42 of the clocks, vector instructions issue in 0.52 to 0.59, and the clock falls with
// a launch's length: 2.35 GHz at 45 us, 2.0 to 2.2 at 150 to 650, 1.86 at 1.2 ms.
//
// 256 rows x 64 tokens.  As in the 64-column tile a wavefront sums group w % 4 of every chunk of
// 256, four 16-wide products a group in the same order of k, scaled into its accumulators group by
// group; here it holds 128 rows x 64 tokens (RB = 4 row blocks), half w / 4 of the tile, so a lookup
// serves 64 tokens, x is read from LDS once for 128 rows, and a chunk is 32 products of 32 clocks a
// wavefront between barriers.  Tokens are the rows of the result: a lane holds one weight row's column
// and its scale.  PAIR: row blocks alternate between gate and up.
//
// Order inside a chunk: vector instructions run beside a matrix instruction if they stand between two of them
// (up to six cost nothing; eight products in a row and then their scaling cost both times).  A unit is
// the four products of 32 rows x 32 tokens; between them stand the scaling of the unit before and, in every
// second unit, the lookups of the next row block, each into the operand register its product has just read
// for the last time.  The order is pinned (sched_barrier): the compiler pulls the units apart again.
//
// Codes: a lane pair fetches the 32 bytes of a row's group; two neighbouring rows' fetches are handed to the
// lanes that multiply them by two lane exchanges (hand_over; on their own no faster than ds_bpermute, which is 6
// clocks of LDS each).  x straight to LDS in 128-byte rows (a token's group), 16-byte pieces XORed with the row's low
// bits, and so the scales.  Flat loads to LDS in flight turn every wait for a register into a wait for all of
// them: codes, x and scales have half a chunk or more to arrive, which no launch here was seen to wait for
// (without any of the loads the loop takes as long).
template <bool PAIR>
__global__ __launch_bounds__(kPromptThreads) void prompt_gemm(const PromptArgs a) {
  extern __shared__ __align__(16) uint32_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave & 3, half = wave >> 2;
  const int r = lane & 31, h = lane >> 5;
  const uint32_t lane4 = static_cast<uint32_t>(lane) * 4;

  // each XCD takes a run of tiles, token tiles fastest: workgroups that share weights meet in one L2
  const int total = static_cast<int>(gridDim.x);
  const int xcd = static_cast<int>(blockIdx.x) & 7;
  const int tile = xcd * (total >> 3) + min(xcd, total & 7) + (static_cast<int>(blockIdx.x) >> 3);
  const int tn = tile % a.tiles_n;
  const int tms = tile / a.tiles_n;
  const int tm = tms % a.tiles_m;
  const int split = tms / a.tiles_m;
  const int c_lo = split * a.split_chunks;
  const int c_hi = min(c_lo + a.split_chunks, a.chunks);
  const int tok0 = tn * kWindow;
  const int groups = a.chunks * 4;

  // row of a matrix for row `lr` of the tile (clamped: rows past the end are not stored)
  auto out_row = [&](int lr) {
    if constexpr (PAIR) {
      return tm * (kTileRows / 2) + (lr >> 6) * 32 + (lr & 31);
    } else {
      return tm * kTileRows + lr;
    }
  };
  auto locate = [&](int lr, int &mat) {
    int row = min(out_row(lr), a.M - 1);
    if constexpr (PAIR) {
      mat = (lr >> 5) & 1;
    } else {
      mat = row >= a.first[2] ? 2 : (row >= a.first[1] ? 1 : 0);
      row -= a.first[mat];
    }
    return row;
  };
  const uint8_t *wp[kBlocks];
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
    int mat;
    const int row = locate(half * (kTileRows / 2) + (b >> 1) * 64 + (lane & ~1) + (b & 1), mat);
    const uint8_t *base = mat == 0 ? a.packed[0] : (mat == 1 ? a.packed[1] : a.packed[2]);
    wp[b] = base + static_cast<size_t>(row) * groups * 32 + g * 32 + (lane & 1) * 16;
  }
  const uint16_t *sp;
  {
    int mat;
    const int row = locate(tid >> 1, mat);
    const uint16_t *base = mat == 0 ? a.scale[0] : (mat == 1 ? a.scale[1] : a.scale[2]);
    sp = base + static_cast<size_t>(row) * groups + (tid & 1) * 2;
  }
  const bool odd = (lane & 1) != 0;
  const uint16_t *xp =
      a.x + static_cast<size_t>(tok0 + wave * 8 + (lane >> 3)) * a.K + ((lane & 7) ^ (lane >> 3)) * 8;

  auto load_x = [&](int c, int buf) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {  // group p of the chunk, tokens 8 wave .. + 8
      load_to_lds16(xp + c * kChunk + p * kGroup,
                    static_cast<uint32_t>(kXAddr + buf * kXStage + p * (kWindow * 128) + wave * 1024));
    }
  };
  uint4 cw[2];
  auto load_w = [&](int c, int b) { cw[b & 1] = *reinterpret_cast<const uint4 *>(wp[b] + static_cast<size_t>(c) * 128); };
  auto load_s = [&](int c, int buf) {
    load_to_lds4(sp + c * 4, static_cast<uint32_t>(kScaleAddr + buf * kScaleStage + wave * 256));
  };
  // x of row 2 i and y of row 2 i + 1 hold half `lane & 1` of their rows' groups; afterwards lane (r, h) has half
  // h of row r in lo and of row 32 + r in hi
  auto hand_over = [&](uint32_t x, uint32_t y, uint32_t &lo, uint32_t &hi) {
    const uint32_t xn = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), kDppQuadXor1, 0xF, 0xF, true));
    const uint32_t yn = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(y), kDppQuadXor1, 0xF, 0xF, true));
    const auto p = __builtin_amdgcn_permlane32_swap(odd ? yn : x, odd ? y : xn, false, false);
    lo = p[0];
    hi = p[1];
  };
  load_x(c_lo, 0);
  load_s(c_lo, 0);
  load_w(c_lo, 0);
  load_w(c_lo, 1);
  // the table, its low levels literals (a byte a turn with two loads each, 4 us a workgroup)
  {
    uint32_t hi[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      hi[i] = bf16_bits_rne(kLutBits[wave + i * 8]) << 16;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int l = 0; l < 16; ++l) {
        smem[(16 * (wave + i * 8) + l) * 64 + lane] = hi[i] | bf16_bits_rne(kLevelBits[l]);
      }
    }
  }
  lds_loads_done();
  __syncthreads();

  F32x16 acc[kBlocks][2];
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[b][t][v] = 0.f;
      }
    }
  }
  uint32_t codes[2][4];
  Bf16x8 wf[4];
  auto hand_over_pair = [&]() {
    hand_over(cw[0].x, cw[1].x, codes[0][0], codes[1][0]);
    hand_over(cw[0].y, cw[1].y, codes[0][1], codes[1][1]);
    hand_over(cw[0].z, cw[1].z, codes[0][2], codes[1][2]);
    hand_over(cw[0].w, cw[1].w, codes[0][3], codes[1][3]);
  };
  uint32_t at[4];  // table addresses of one of a block's four operands
  auto address = [&](int b, int j, int k) {
    constexpr uint32_t sel = 0x0C0C0400u;
    at[k] = __builtin_amdgcn_perm(codes[b & 1][j], lane4, sel + (static_cast<uint32_t>(k) << 8));
  };
  auto look_up = [&](int j) {
    const Raw16 f = {lds0_u32(at[0]), lds0_u32(at[1]), lds0_u32(at[2]), lds0_u32(at[3])};
    wf[j] = __builtin_bit_cast(Bf16x8, f);
  };
  // the first block's operands, as every block before leaves them
  hand_over_pair();
  load_w(c_lo, 2);
  load_w(c_lo, 3);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      address(0, j, k);
    }
    look_up(j);
  }
  F32x16 d[2];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    d[1][v] = 0.f;
  }
  float s_old = 0.f;
  int buf = 0;
  for (int c = c_lo; c < c_hi; ++c) {
    // the last chunk asks for its own x again and drops it: requests behind a branch are waited for
    const int next = min(c + 1, c_hi - 1);
    asm volatile("" ::: "memory");
    load_x(next, buf ^ 1);
    load_s(next, buf ^ 1);
    asm volatile("" ::: "memory");
    Bf16x8 xf[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t at = static_cast<uint32_t>(kXAddr + buf * kXStage + g * (kWindow * 128) + (t * 32 + r) * 128 +
                                                  (((4 * h + j) ^ (r & 7)) << 4));
        xf[t][j] = __builtin_bit_cast(Bf16x8, lds0_u128(at));
      }
    }
    const uint32_t s_at = static_cast<uint32_t>(kScaleAddr + buf * kScaleStage + (half * (kTileRows / 2) + r) * 8 + g * 2);
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
      const float s_now = f16_to_f32(*reinterpret_cast<const __attribute__((address_space(3))) uint16_t *>(s_at + b * 256));
      if (b & 1) {  // the codes of the next two blocks; their registers are asked for again behind it
        __builtin_amdgcn_sched_barrier(0);
        hand_over_pair();
        __builtin_amdgcn_sched_barrier(0);
        load_w(next, b == 1 ? 0 : 2);
        load_w(next, b == 1 ? 1 : 3);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          __builtin_amdgcn_sched_barrier(0);
          if (j == 0) {
            F32x16 z;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              z[v] = 0.f;
            }
            d[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[t][j], wf[j], z, 0, 0, 0);
          } else {
            d[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[t][j], wf[j], d[t], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          const int nb = (b + 1) & 3;
          if (t == 0 && j == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              address(nb, 0, k);
            }
          }
          if (t == 1) {
            look_up(j);
          }
          __builtin_amdgcn_sched_barrier(0);
          if (t == 1 && j < 3) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              address(nb, j + 1, k);
            }
          }
          // unit before: (b, 0) beside (b, 1), (b - 1, 1) beside (b, 0)
          const int pb = t == 1 ? b : (b + 3) & 3, pt = t ^ 1;
          const float s = t == 1 ? s_now : s_old;
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            if (v * 3 / 16 == j - 1) {
              acc[pb][pt][v] = fmaf(s, d[pt][v], acc[pb][pt][v]);
            }
          }
        }
      }
      s_old = s_now;
    }
    __builtin_amdgcn_sched_barrier(0);
    // the next chunk's x and scales are the oldest requests but the four of codes since
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __syncthreads();
    buf ^= 1;
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    acc[kBlocks - 1][1][v] = fmaf(s_old, d[1][v], acc[kBlocks - 1][1][v]);
  }
  lds_loads_done();
  __syncthreads();

  // The four wavefronts' sums of every output meet in LDS (the table and x are done with), two row blocks at
  // a time.  There lanes 4 i .. 4 i + 3 of a result register are four successive rows of one token: a thread
  // adds the four sums of these, in group order, and stores them as one vector (a row of one token a lane and
  // four bytes a store, the stores took as long as two chunks).
  float *sums = reinterpret_cast<float *>(smem);
  static_assert(2 * 2 * 8 * 16 * kWave * 4 <= kScaleAddr, "the sums of two row blocks fit");
  const size_t row_floats = static_cast<size_t>(PAIR ? 2 * a.M : a.M);
  const int quad = (tid & 7) * 4, at_h = (tid >> 3) & 1, at_v = (tid >> 4) & 15;  // rows, and the token's place
  const int at_half = tid >> 8;
#pragma unroll
  for (int pass = 0; pass < kBlocks / 2; ++pass) {
    if (pass > 0) {
      __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          sums[(((b * 2 + t) * 8 + wave) * 16 + v) * kWave + lane] = acc[2 * pass + b][t][v];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      F32x4 o[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        o[b] = F32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const F32x4 part = *reinterpret_cast<const F32x4 *>(
              sums + (((b * 2 + t) * 8 + 4 * at_half + q) * 16 + at_v) * kWave + at_h * 32 + quad);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            o[b][e] += part[e];
          }
        }
      }
      const size_t tok = static_cast<size_t>(tok0 + t * 32 + 8 * (at_v >> 2) + 4 * at_h + (at_v & 3));
      if constexpr (PAIR) {
        const int row = out_row(at_half * (kTileRows / 2) + 2 * pass * 32 + quad);
        if (row < a.M) {
          if (a.part != nullptr) {
            float *dst = a.part + (static_cast<size_t>(split) * a.N + tok) * row_floats + row;
            *reinterpret_cast<F32x4 *>(dst) = o[0];
            *reinterpret_cast<F32x4 *>(dst + a.M) = o[1];
          } else {
            uint32_t out[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              out[e] = swiglu_bf16(o[0][e], o[1][e]);
            }
            *reinterpret_cast<uint2 *>(a.y + tok * a.M + row) = make_uint2(out[0] | (out[1] << 16), out[2] | (out[3] << 16));
          }
        }
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int row = out_row(at_half * (kTileRows / 2) + (2 * pass + b) * 32 + quad);
          if (row < a.M) {
            if (a.part != nullptr) {
              *reinterpret_cast<F32x4 *>(a.part + (static_cast<size_t>(split) * a.N + tok) * row_floats + row) = o[b];
            } else {
              uint32_t out[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                out[e] = f32_to_bf16(o[b][e]);
                if (a.bias != nullptr) {
                  out[e] = f32_to_bf16(bf16_to_f32(static_cast<uint16_t>(out[e])) + bf16_to_f32(a.bias[row + e]));
                }
              }
              *reinterpret_cast<uint2 *>(a.y + tok * a.M + row) = make_uint2(out[0] | (out[1] << 16), out[2] | (out[3] << 16));
            }
          }
        }
      }
    }
  }
}

__device__ __forceinline__ F32x4 sum_in_order(const float *p, int splits, size_t stride) {
  F32x4 s = *reinterpret_cast<const F32x4 *>(p);
#pragma unroll 4
  for (int j = 1; j < splits; ++j) {
    const F32x4 v = *reinterpret_cast<const F32x4 *>(p + j * stride);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[e] += v[e];
    }
  }
  return s;
}

// The splits of a product, four features a thread: bf16 of the sum (+ bias), or silu(gate) * up.
template <bool PAIR>
__global__ __launch_bounds__(256) void prompt_reduce(const float *__restrict__ part, int splits, int64_t quads, int M,
                                                     int64_t count, const uint16_t *__restrict__ bias,
                                                     uint16_t *__restrict__ y) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (q >= quads) {
    return;
  }
  const int64_t at = q * 4;
  const int m = static_cast<int>(at % M);
  uint16_t o[4];
  if constexpr (PAIR) {
    const float *p = part + (at / M) * 2 * M + m;
    const F32x4 g = sum_in_order(p, splits, 2 * count), u = sum_in_order(p + M, splits, 2 * count);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = swiglu_bf16(g[e], u[e]);
    }
  } else {
    const F32x4 s = sum_in_order(part + at, splits, count);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = f32_to_bf16(s[e]);
      if (bias != nullptr) {
        o[e] = f32_to_bf16(bf16_to_f32(o[e]) + bf16_to_f32(bias[m + e]));
      }
    }
  }
  *reinterpret_cast<uint2 *>(y + at) =
      make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16), o[2] | (static_cast<uint32_t>(o[3]) << 16));
}

// lane Q of every four
template <int Q>
__device__ __forceinline__ float of_quad(float v) {
  return dpp_f32<Q * 0x55>(v);
}

// One workgroup a token: x += bf16(sum of the splits) (+ bias), and with norm_w h = RMSNorm(x).  Bound: the
// partials it reads.  A thread takes four neighbouring features in each of four passes, so a wavefront's
// requests are whole lines and all of a split's leave together (with 16 neighbouring features a thread 1728
// tokens of 5120 behind three splits and behind six took 59 + 121 us, 83 in all so; 512 tokens 13, 11).  The
// squares are added as the 64-column tile's column sums and rms_cols add them: a block of 16 rows in the order 0 4 1 5 2 6 3 7 8 12 9 13 10 14 11 15 (four lanes hold it, each
// adds all of it), sixteen chains of every sixteenth block, the chains in order.
__global__ __launch_bounds__(1024) void prompt_add_rms(const float *__restrict__ part, int splits, size_t stride, int M,
                                                       const uint16_t *__restrict__ bias, uint16_t *__restrict__ x,
                                                       const uint16_t *__restrict__ norm_w, float eps,
                                                       uint16_t *__restrict__ h) {
  __shared__ float block_sum[1024], chain[16];
  const int tid = threadIdx.x, threads = blockDim.x, blocks = M / 16;
  const size_t row = static_cast<size_t>(blockIdx.x) * M;
  float f[4][4];
  F32x4 s[4];
  uint2 packed[4];
  // requests without a branch: features past the last are its again, and dropped
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int m = min((p * threads + tid) * 4, M - 4);
    packed[p] = *reinterpret_cast<const uint2 *>(x + row + m);
    s[p] = *reinterpret_cast<const F32x4 *>(part + row + m);
  }
#pragma unroll 4
  for (int j = 1; j < splits; ++j) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int m = min((p * threads + tid) * 4, M - 4);
      const F32x4 v = *reinterpret_cast<const F32x4 *>(part + j * stride + row + m);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[p][e] += v[e];
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int quad = p * threads + tid, m = quad * 4;  // (whole blocks of four quads are in or out)
    if (m >= M) {
      continue;
    }
    const float was[4] = {bf16_lo(packed[p].x), bf16_hi(packed[p].x), bf16_lo(packed[p].y), bf16_hi(packed[p].y)};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float t = bf16_to_f32(f32_to_bf16(s[p][e]));
      if (bias != nullptr) {
        t = bf16_to_f32(f32_to_bf16(t + bf16_to_f32(bias[m + e])));
      }
      f[p][e] = bf16_to_f32(f32_to_bf16(was[e] + t));
    }
    *reinterpret_cast<uint2 *>(x + row + m) = make_uint2(f32x2_to_bf16x2(f[p][0], f[p][1]), f32x2_to_bf16x2(f[p][2], f[p][3]));
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = of_quad<0>(f[p][e]), b = of_quad<1>(f[p][e]);
      sum = __fadd_rn(sum, __fmul_rn(a, a));
      sum = __fadd_rn(sum, __fmul_rn(b, b));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = of_quad<2>(f[p][e]), b = of_quad<3>(f[p][e]);
      sum = __fadd_rn(sum, __fmul_rn(a, a));
      sum = __fadd_rn(sum, __fmul_rn(b, b));
    }
    if ((tid & 3) == 0) {
      block_sum[quad >> 2] = sum;
    }
  }
  if (norm_w == nullptr) {
    return;
  }
  __syncthreads();
  if (tid < 16) {
    float t = 0.f;
    for (int i = tid; i < blocks; i += 16) {
      t += block_sum[i];
    }
    chain[tid] = t;
  }
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    t += chain[i];
  }
  const float inv = rsqrtf(t / static_cast<float>(M) + eps);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int m = (p * threads + tid) * 4;
    if (m >= M) {
      continue;
    }
    float out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      out[e] = (bf16_to_f32(norm_w[m + e]) * f[p][e]) * inv;
    }
    *reinterpret_cast<uint2 *>(h + row + m) = make_uint2(f32x2_to_bf16x2(out[0], out[1]), f32x2_to_bf16x2(out[2], out[3]));
  }
}

// RMSNorm of rows nobody left sums for (the embedding's), squares added as rms_cols adds those of a
// 64-column tile it reads itself: 128 chains of every 128th feature, eight neighbouring chains by
// halves, the sixteen results in order.
__global__ __launch_bounds__(128) void prompt_rms(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
                                                  uint16_t *__restrict__ h, int M, float eps) {
  __shared__ float part[16];
  const uint16_t *row = x + static_cast<size_t>(blockIdx.x) * M;
  uint16_t *dst = h + static_cast<size_t>(blockIdx.x) * M;
  float ss = 0.f;
  for (int k = threadIdx.x; k < M; k += 128) {
    const float v = bf16_to_f32(row[k]);
    ss = fmaf(v, v, ss);
  }
  ss += __shfl_down(ss, 4, 8);
  ss += __shfl_down(ss, 2, 8);
  ss += __shfl_down(ss, 1, 8);
  if ((threadIdx.x & 7) == 0) {
    part[threadIdx.x >> 3] = ss;
  }
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    t += part[i];
  }
  const float inv = rsqrtf(t / static_cast<float>(M) + eps);
  for (int k = threadIdx.x; k < M; k += 128) {
    dst[k] = f32_to_bf16((bf16_to_f32(w[k]) * bf16_to_f32(row[k])) * inv);
  }
}

// Rotate-half RoPE of rows [q | k | v] and the cache write: rope_kv_cols (dv2_prefill.hip) on
// token-major data, the same arithmetic.  A thread takes W dims of a head's lower half and their
// partners.
template <int W>
__global__ __launch_bounds__(256) void rope_kv_rows(const uint16_t *__restrict__ qkv, int n, int n_q, int n_kv, int hd,
                                                    int start, uint16_t *__restrict__ q_out,
                                                    uint16_t *__restrict__ k_cache, uint16_t *__restrict__ v_cache,
                                                    const uint16_t *__restrict__ cos, const uint16_t *__restrict__ sin) {
  const int half = hd / 2;
  const int per_head = half / W;
  const int64_t items = static_cast<int64_t>(n) * (n_q + n_kv) * per_head;
  for (int64_t it = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; it < items;
       it += static_cast<int64_t>(gridDim.x) * 256) {
    const int d0 = static_cast<int>(it % per_head) * W;
    const int hid = static_cast<int>((it / per_head) % (n_q + n_kv));
    const int64_t tok = it / per_head / (n_q + n_kv);
    const uint16_t *src = qkv + (tok * (n_q + 2 * n_kv) + hid) * hd + d0;
    const int64_t pos = start + tok;
    const uint16_t *c = cos + pos * hd + d0, *s = sin + pos * hd + d0;
    uint16_t lo[W], hi[W];
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const float a0 = bf16_to_f32(src[e]), a1 = bf16_to_f32(src[half + e]);
      lo[e] = f32_to_bf16(a0 * bf16_to_f32(c[e]) + (-a1) * bf16_to_f32(s[e]));
      hi[e] = f32_to_bf16(a1 * bf16_to_f32(c[half + e]) + a0 * bf16_to_f32(s[half + e]));
    }
    uint16_t *dst = q_out + (tok * n_q + hid) * hd + d0;
    if (hid >= n_q) {
      const int64_t at = (pos * n_kv + (hid - n_q)) * hd + d0;
      dst = k_cache + at;
      const uint16_t *v = src + static_cast<int64_t>(n_kv) * hd;
#pragma unroll
      for (int e = 0; e < W; ++e) {
        v_cache[at + e] = v[e];
        v_cache[at + half + e] = v[half + e];
      }
    }
#pragma unroll
    for (int e = 0; e < W; ++e) {
      dst[e] = lo[e];
      dst[half + e] = hi[e];
    }
  }
}

// Checks shared by the products; fills what the matrices decide.
int prompt_args(const chr_nf4_dev_t *w, int32_t n_mats, bool pair, int32_t N, PromptArgs &a) {
  if (w == nullptr) {
    return -1;
  }
  if (N < kWindow || N % kWindow != 0) {
    return -2;
  }
  if (n_mats < 1 || n_mats > kPromptMats || (pair && (n_mats != 2 || w[0].M != w[1].M))) {
    return -3;
  }
  int64_t rows = 0;
  for (int i = 0; i < n_mats; ++i) {
    if (w[i].M < 1 || w[i].K < 1 || w[i].packed == nullptr || w[i].scale == nullptr || w[i].K != w[0].K) {
      return -3;
    }
    if (!k_pad_ok(w[i].K, w[i].K_pad)) {
      return -4;
    }
    if (!aligned16(w[i].packed) || (reinterpret_cast<uintptr_t>(w[i].scale) & 7u) != 0) {
      return -5;
    }
    a.packed[i] = w[i].packed;
    a.scale[i] = w[i].scale;
    a.first[i] = static_cast<int>(rows);
    rows += w[i].M;
  }
  a.split_chunks = window64_chunks(w, n_mats);
  if (a.split_chunks < 1 || w[0].K % kChunk != 0 || rows > INT32_MAX / 2 || rows % 4 != 0 || w[0].M % 4 != 0) {
    return -3;
  }
  for (int i = n_mats; i <= kPromptMats; ++i) {
    a.first[i] = static_cast<int>(rows);
  }
  a.M = pair ? w[0].M : static_cast<int>(rows);
  a.N = N;
  a.K = w[0].K;
  a.chunks = a.K / kChunk;
  a.tiles_m = (a.M + kTileRows / (pair ? 2 : 1) - 1) / (kTileRows / (pair ? 2 : 1));
  a.tiles_n = N / kWindow;
  return 0;
}

int prompt_splits(const PromptArgs &a) { return (a.chunks + a.split_chunks - 1) / a.split_chunks; }

template <bool PAIR>
int prompt_launch(const PromptArgs &a, hipStream_t st) {
  const int64_t grid = static_cast<int64_t>(a.tiles_m) * a.tiles_n * prompt_splits(a);
  if (grid > INT32_MAX) {
    return -3;
  }
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(&prompt_gemm<PAIR>), hipFuncAttributeMaxDynamicSharedMemorySize,
                          kPromptLds) != hipSuccess) {
    (void)hipGetLastError();
    return -6;
  }
  prompt_gemm<PAIR><<<dim3(static_cast<unsigned>(grid)), dim3(kPromptThreads), kPromptLds, st>>>(a);
  return launch_rc();
}

}  // namespace
}  // namespace chr

using namespace chr;

extern "C" int64_t chr_dv2_prompt_ws(const chr_nf4_dev_t *w, int32_t n_mats, int32_t kind, int32_t N) {
  PromptArgs a{};
  if (kind < 0 || kind > 2 || prompt_args(w, n_mats, kind == 1, N, a) != 0) {
    return -1;
  }
  const int splits = prompt_splits(a);
  return splits == 1 && kind != 2 ? 0 : static_cast<int64_t>(splits) * N * a.M * (kind == 1 ? 2 : 1);
}

extern "C" int chr_dv2_prompt_gemm(const chr_nf4_dev_t *w, int32_t n_mats, int32_t swiglu, const void *x, int32_t N,
                                   void *y, float *ws, int64_t ws_floats, const void *bias, void *stream) {
  if (x == nullptr || y == nullptr) {
    return -1;
  }
  PromptArgs a{};
  const bool pair = swiglu != 0;
  if (const int rc = prompt_args(w, n_mats, pair, N, a)) {
    return rc;
  }
  if (pair && bias != nullptr) {
    return -3;
  }
  const int splits = prompt_splits(a);
  const int64_t need = chr_dv2_prompt_ws(w, n_mats, pair ? 1 : 0, N);
  if (!aligned16(x) || !aligned16(y) || (need > 0 && !aligned16(ws))) {
    return -5;
  }
  if (need > 0 && (ws == nullptr || ws_floats < need)) {
    return -7;
  }
  a.x = static_cast<const uint16_t *>(x);
  a.y = static_cast<uint16_t *>(y);
  a.bias = static_cast<const uint16_t *>(bias);
  a.part = need > 0 ? ws : nullptr;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int rc = pair ? prompt_launch<true>(a, st) : prompt_launch<false>(a, st);
  if (rc != 0 || need == 0) {
    return rc;
  }
  const int64_t count = static_cast<int64_t>(N) * a.M;
  const dim3 grid(static_cast<unsigned>((count / 4 + 255) / 256)), block(256);
  if (pair) {
    prompt_reduce<true><<<grid, block, 0, st>>>(a.part, splits, count / 4, a.M, count, nullptr, a.y);
  } else {
    prompt_reduce<false><<<grid, block, 0, st>>>(a.part, splits, count / 4, a.M, count, a.bias, a.y);
  }
  return launch_rc();
}

extern "C" int chr_dv2_prompt_add_rms(const chr_nf4_dev_t *w, const void *x, int32_t N, void *residual, const void *bias,
                                      const void *norm_w, float eps, void *h, float *ws, int64_t ws_floats,
                                      void *stream) {
  if (x == nullptr || residual == nullptr || (norm_w != nullptr && h == nullptr)) {
    return -1;
  }
  PromptArgs a{};
  if (const int rc = prompt_args(w, 1, false, N, a)) {
    return rc;
  }
  if (a.M % 16 != 0 || a.M / 16 > 1024) {
    return -3;
  }
  const int64_t need = chr_dv2_prompt_ws(w, 1, 2, N);
  if (!aligned16(x) || !aligned16(residual) || !aligned16(h) || !aligned16(ws)) {
    return -5;
  }
  if (ws == nullptr || ws_floats < need) {
    return -7;
  }
  a.x = static_cast<const uint16_t *>(x);
  a.part = ws;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (const int rc = prompt_launch<false>(a, st)) {
    return rc;
  }
  const int threads = (a.M / 16 + kWave - 1) / kWave * kWave;
  prompt_add_rms<<<dim3(static_cast<unsigned>(N)), dim3(static_cast<unsigned>(threads)), 0, st>>>(
      ws, prompt_splits(a), static_cast<size_t>(N) * a.M, a.M, static_cast<const uint16_t *>(bias),
      static_cast<uint16_t *>(residual), static_cast<const uint16_t *>(norm_w), eps, static_cast<uint16_t *>(h));
  return launch_rc();
}

extern "C" int chr_dv2_prompt_rms(const void *x, const void *w, void *h, int32_t N, int32_t M, float eps, void *stream) {
  if (x == nullptr || w == nullptr || h == nullptr) {
    return -1;
  }
  if (N < 1 || M < 1) {
    return -3;
  }
  prompt_rms<<<dim3(static_cast<unsigned>(N)), dim3(128), 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(w), static_cast<uint16_t *>(h), M, eps);
  return launch_rc();
}

extern "C" int chr_dv2_rope_kv_rows(const void *qkv, void *q_out, int32_t N, int32_t n_q, int32_t n_kv, int32_t hd,
                                    int32_t start, int32_t max_seq, void *k_cache, void *v_cache, const void *cos,
                                    const void *sin, void *stream) {
  if (qkv == nullptr || q_out == nullptr || k_cache == nullptr || v_cache == nullptr || cos == nullptr || sin == nullptr) {
    return -1;
  }
  if (N < 1) {
    return -2;
  }
  if (n_q < 1 || n_kv < 1 || hd < 2 || (hd & 1) != 0 || max_seq < 1 || start < 0 || N > max_seq - start) {
    return -3;
  }
  const bool quads = hd % 8 == 0;
  const int64_t items = static_cast<int64_t>(N) * (n_q + n_kv) * (hd / 2 / (quads ? 4 : 1));
  const dim3 grid(static_cast<unsigned>(items / 256 < 65535 ? items / 256 + 1 : 65536)), block(256);
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto run = [&](auto kernel) {
    kernel<<<grid, block, 0, st>>>(static_cast<const uint16_t *>(qkv), N, n_q, n_kv, hd, start,
                                   static_cast<uint16_t *>(q_out), static_cast<uint16_t *>(k_cache),
                                   static_cast<uint16_t *>(v_cache), static_cast<const uint16_t *>(cos),
                                   static_cast<const uint16_t *>(sin));
  };
  if (quads) {
    run(rope_kv_rows<4>);
  } else {
    run(rope_kv_rows<1>);
  }
  return launch_rc();
}
