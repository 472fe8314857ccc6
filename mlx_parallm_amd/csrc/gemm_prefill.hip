// gemm_prefill.hip -- MFMA tile GEMM for the prefill call of generate_step (L > 1 tokens per row):
//   C[M][N] = X[M][K] . W[N][K]^T   (nn.Linear on (B, L, H) activations: llama.py:93,143,165)
// plus the row-wise RMSNorm that feeds it (llama.py:187,189) and the residual / SwiGLU epilogues.
// 16-bit activations, dense 16-bit weights in the tile-major layout of repack.hip.  The decode
// kernels (gemv_mfma.hip) stream W once per <= 16 rows; here a 128 x 128 output tile re-uses
// every weight fragment over 128 rows, which makes the call MFMA-bound instead of HBM-bound.
//
// Block = 256 threads = 4 waves as 2 (M) x 2 (N); wave tile 64 x 64 = 4 x 4 MFMA tiles
// (v_mfma_f32_16x16x32, 64 accumulator registers); K step 64.
//   * X tile (128 x 64) goes global -> registers -> LDS, rows padded to 144 B so that the 16 lanes
//     of an A-fragment read (16 consecutive rows, one 16-B chunk each) hit 16 distinct bank groups;
//     double-buffered, the next tile's global loads are issued before the current tile's MFMAs.
//   * W fragments come straight from global memory in MFMA order: in the tile-major layout the
//     fragment of (16 rows, 32 k) is one contiguous KiB, lane l at 16 l -- no LDS, no transpose.
//     The next step's 8 fragments are prefetched into a second register set.
//   * SwiGLU: a wave's four N tiles are two gate tiles and the two matching up tiles, so
//     silu(gate) * up happens in registers.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <type_traits>

#include "kernels.h"

namespace mi {

int gemv_cu_count();      // gemv_mfma.hip

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#ifndef MI_GEMM_VARIANT
#define MI_GEMM_VARIANT 0       // A/B experiments (tools/debug/gemm_ab.py); 0 = the shipped kernel
#endif
constexpr int BM = 128, BN = 128, BK = 64;
constexpr int LDA = 72;   // LDS row stride in elements (144 B)

template <typename T>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (std::is_same<T, bf16>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

struct GemmParams {
  const void* x; int ldx; int M;
  const void* w; int N, K;          // W tile-major; N = rows of W (SWIGLU: gate rows = N/2); K = its reduction length
  int ka;                           // reduction length of x: K, or K/2 when W is a [hi | lo] pair (x is walked twice)
  int kw;                           // reduction length of W (its row-tile stride): K, or K/3 when x is a [hi | mid | lo]
                                    // triple of float32 activations (W is walked three times).  k step t multiplies
                                    // x[.., t mod ka] with W[.., t mod kw]; with ka = 3 K0, kw = 2 K0 the 6 K0 steps meet
                                    // every (x part, W part) pair once.
  int out32;                        // outputs / residual stream are float32 (PagedKVCache mode), no 16-bit rounding
  int rnd;                          // .. but for a plain store with logical rounding (layer 0 of that mode: RND_*)
  int strips;                       // rows of the outputs (and the residual) are whole, aligned 16-byte pieces
  int split_out;                    // .. or a SwiGLU stored as two bf16 terms (256 x 256 LDS-DMA tile only)
  int epi; void* out; int ldo; void* resid; int pair_offset;
  Glu glu; int silu_cols;
  // 128 x 128 tile only: K split over gridDim.z workgroups when the (M, N) grid alone leaves most CUs idle (a prompt of a
  // few hundred tokens against N = 4096: 32 x 2..8 blocks); slice z leaves its float32 partial tile in ws[z][M][N] and
  // splitk_epilogue_kernel adds the slices in order and applies the epilogue
  int ksplit; float* ws;
  // codes form, K slices of the last tiles alone: `mb` row blocks (0: the plain grid); the tiles from `tail` on (row blocks fastest) are ksplit workgroups
  // each, which leave their accumulators in ws[tile][slice] for tail_reduce_kernel
  int mb, tail;
  // grouped form (GroupedGemm, kernels.h)
  const int32_t* tiles; const int32_t* x_rows; const int32_t* out_rows; int groups;
  const void* w_last; int N_last, K_last;
  // codes form (gemm_codes256_kernel): w = the codes as 16-bit integers; scales [N/16][G][16], G = kw / 64; the group sums of x
  // [M][kb] and the biases (tile-major, kb columns), whose product follows the K steps
  const float* sc; const void* xs; const void* wb; int G, kb;
};

// the epilogues in float32 storage (PagedKVCache mode after layer 0: every op produces a float32 array)
__device__ __forceinline__ float glu32(const Glu& c, float gt, float up) {
  if (c.kind != GLU_SILU) return glu_f(c, gt, up);
  const float sig = 1.0f / (1.0f + expf(-gt));
  const float sl = gt * sig;
  return sl * up;
}
__device__ __forceinline__ void epi32_swiglu(const GemmParams& p, int m, int n, float gt, float up) {
  ((float*)p.out)[(size_t)m * p.ldo + n] = glu32(p.glu, gt, up);
}
__device__ __forceinline__ void epi32_plain(const GemmParams& p, int m, int n, float y) {
  if (p.epi == EPI_STORE) ((float*)p.out)[(size_t)m * p.ldo + n] = y;
  else { float* h = (float*)p.resid; h[(size_t)m * p.ldo + n] = h[(size_t)m * p.ldo + n] + y; }
}

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// grid: (n blocks, m blocks).  SWIGLU: a block covers 64 gate columns + the 64 matching up columns.
// grouped form: the matrix and the rows of tile bm of the device-resident table; false: no such tile, or no columns from n0 on
template <typename AT, bool SWIGLU>
__device__ __forceinline__ bool group_of_tile(GemmParams& p, int bm, int n0, int& place0) {
  if (bm >= p.tiles[0]) return false;
  const int32_t* t = p.tiles + 8 + 4 * bm;
  const int grp = t[0];
  place0 = t[1]; p.M = t[2];
  if (grp == p.groups) { p.w = p.w_last; p.N = p.N_last; p.K = p.ka = p.kw = p.K_last; }
  else p.w = (const char*)p.w + (size_t)grp * p.N * p.K * sizeof(AT);
  if constexpr (SWIGLU) p.pair_offset = p.N / 2;
  return n0 < (SWIGLU ? p.pair_offset : p.N);
}

// GROUPED: blockIdx.x = tile of the device-resident table; every group of rows has its own matrix (GroupedGemm, kernels.h)
// FOLD: the accumulators are added to a second set every three K steps, i.e. no float32 chain is longer than six MFMAs + K / 192
// additions.  For outputs that are ROUNDED to 16 bits where an exact computation rounds too (layer 0 of the float32-cache mode): the
// longer the chain, the more values round the other way (mean |logprob - exact| of three recorded float32-cache cases: streaming
// kernel 1.64 / 1.27 / 2.08e-4, the 256 x 256 tile's one chain over K 2.02 / 1.74 / 2.53e-4, here 1.52 / 1.04 / 1.98e-4).  8 x 1024 rows
// of Mistral-7B's q|k|v: 0.9 ms against 0.4 on the 256 x 256 tile and 4.6 streaming.
// LOGITS (here and in the 256 x 256 kernels): plain float32 stores of values rounded to AT.  A form of its own: p.rnd asked per element cost every
// call of the kernels (one round of 256 workgroups, 8192 x 2048 outputs, 67.7 -> 76.0 us).
template <typename AT, bool SWIGLU, bool GROUPED = false, bool FOLD = false, bool LOGITS = false>
__global__ __launch_bounds__(256) void gemm_tile_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(16))) AT As[2][BM][LDA];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int c16 = lane & 15, g = lane >> 4;
  // blockIdx.x = M block (fastest): the blocks that run together share one N block, i.e. the same
  // W tiles, which then stay in the XCD's L2 instead of being re-fetched per block
  const int bm = blockIdx.x, bn = blockIdx.y;
  int m0 = bm * BM, place0 = 0;
  if constexpr (GROUPED) {
    if (!group_of_tile<AT, SWIGLU>(p, bm, bn * (SWIGLU ? 64 : BN), place0)) return;
    m0 = 0;
  }
  const int nk_all = p.K / BK, nkw = p.kw / BK;
  const int ks0 = (int)(((long)blockIdx.z * nk_all) / p.ksplit), ks1 = (int)(((long)(blockIdx.z + 1) * nk_all) / p.ksplit);
  const int nk = ks1;                               // (the loop runs over [ks0, ks1); "nk" bounds the prefetches)
  const AT* x = (const AT*)p.x;

  // W tiles (16 rows each) of this wave's four N tiles
  int wtile[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    if constexpr (!SWIGLU) wtile[nt] = (bn * BN + wn * 64 + nt * 16) / 16;
    else wtile[nt] = (bn * 64 + wn * 32 + (nt & 1) * 16 + (nt >> 1) * p.pair_offset) / 16;
  }
  const int ntiles_w = p.N / 16;

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- X tile loads: 128 rows x 8 chunks of 16 B; thread -> chunks tid, tid+256, ...
  // (straight-line: rows past M read row M - 1 and are zeroed on the way into LDS -- see gemm_tile256_kernel)
  u32x4 areg[4];
  const AT* arow[4];
  bool aok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + 256 * i, row = c >> 3, kq = c & 7;
    aok[i] = m0 + row < p.M;
    int xr = min(m0 + row, p.M - 1);
    if constexpr (GROUPED) { xr += place0; if (p.x_rows != nullptr) xr = p.x_rows[xr]; }
    arow[i] = x + (size_t)xr * p.ldx + kq * 8;
  }
  auto load_a = [&](int ks) {
    const int ka = (ks * BK) % p.ka;
#pragma unroll
    for (int i = 0; i < 4; ++i) areg[i] = *(const u32x4*)(arow[i] + ka);
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + 256 * i, row = c >> 3, kq = c & 7;
      *(u32x4*)&As[buf][row][kq * 8] = aok[i] ? areg[i] : u32x4{0u, 0u, 0u, 0u};
    }
  };
  const bool live = !GROUPED || wm * 64 < p.M;     // (grouped: a short tile leaves half of the waves without rows)
  u32x4 breg[3][4][2];     // [set][n tile][k block]; W fragments are fetched two K steps ahead
  auto load_b = [&](int set, int ks) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int t = min(wtile[nt], ntiles_w - 1);
        const char* blk = (const char*)p.w + ((size_t)t * (p.kw / 32) + (size_t)((ks % nkw) * 2 + kb)) * 1024;
        breg[set][nt][kb] = *(const u32x4*)(blk + lane * 16);
      }
  };

  load_a(ks0);
  load_b(0, ks0);
  if (ks0 + 1 < nk) load_b(1, ks0 + 1);
  store_a(0);
  __syncthreads();

  // the K loop is unrolled by 3 so that the register set of each step is a compile-time index
  auto step = [&](int ks, auto set_tag) {
    constexpr int SET = decltype(set_tag)::value;
    const int cur = (ks - ks0) & 1;
    load_a(min(ks + 1, nk - 1));
    if (live) load_b((SET + 2) % 3, min(ks + 2, nk - 1));
    __builtin_amdgcn_sched_barrier(0);           // the loads stay ahead of this step's MFMAs
    if (live)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      u32x4 af[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) af[mt] = *(const u32x4*)&As[cur][wm * 64 + mt * 16 + c16][kb * 32 + g * 8];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = mfma16<AT>(af[mt], breg[SET][nt][kb], acc[mt][nt]);
    }
    if (ks + 1 < nk) {
      store_a(cur ^ 1);       // buffer cur^1 was last read one step ago; the barrier of that step separates
      __syncthreads();
    }
  };
  f32x4 tot[FOLD ? 4 : 1][FOLD ? 4 : 1];
#pragma unroll
  for (int i = 0; i < (FOLD ? 4 : 1); ++i)
#pragma unroll
    for (int j = 0; j < (FOLD ? 4 : 1); ++j) tot[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int ks = ks0; ks < nk; ks += 3) {
    step(ks, std::integral_constant<int, 0>{});
    if (ks + 1 < nk) step(ks + 1, std::integral_constant<int, 1>{});
    if (ks + 2 < nk) step(ks + 2, std::integral_constant<int, 2>{});
    if constexpr (FOLD) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) { tot[i][j] += acc[i][j]; acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
    }
  }
  if constexpr (FOLD) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = tot[i][j];
  }

  if constexpr (!SWIGLU) {
    if (p.ksplit > 1) {                            // this K slice's partial tile, float32, for splitk_epilogue_kernel
      float* wz = p.ws + (size_t)blockIdx.z * p.M * p.N;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm * 64 + mt * 16 + 4 * g + r;
          if (m >= p.M) continue;
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) {
            const int n = bn * BN + wn * 64 + nt * 16 + c16;
            if (n < p.N) wz[(size_t)m * p.N + n] = acc[mt][nt][r];
          }
        }
      return;
    }
  }

  // ---- epilogue: lane (c16, g) holds C[m = 4g + r][n = c16] of every 16 x 16 tile
  // (var: another unit than silu, or a plain store with silu columns -- asked once, not per element)
  AT* out = (AT*)p.out;
  auto store = [&](auto var) {
    constexpr bool VAR = decltype(var)::value;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      int m = m0 + wm * 64 + mt * 16 + 4 * g + r;
      if (m >= p.M) continue;
      if constexpr (GROUPED) { m += place0; if (p.out_rows != nullptr) m = p.out_rows[m]; }
      if constexpr (SWIGLU) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = bn * 64 + wn * 32 + j * 16 + c16;
          if (n >= p.pair_offset) continue;
          if constexpr (GROUPED) { out[(size_t)m * p.ldo + n] = (AT)(VAR ? glu_f(p.glu, acc[mt][j][r], acc[mt][j + 2][r]) : silu_mul(acc[mt][j][r], acc[mt][j + 2][r])); continue; }
          if (p.out32) { epi32_swiglu(p, m, n, acc[mt][j][r], acc[mt][j + 2][r]); continue; }
          out[(size_t)m * p.ldo + n] = (VAR ? (AT)glu_f(p.glu, acc[mt][j][r], acc[mt][j + 2][r]) : silu16<AT>(acc[mt][j][r], acc[mt][j + 2][r]));
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          const int n = bn * BN + wn * 64 + nt * 16 + c16;
          if (n >= p.N) continue;
          if constexpr (FOLD || LOGITS) { ((float*)p.out)[(size_t)m * p.ldo + n] = LOGITS ? (float)(AT)acc[mt][nt][r] : round_rt(acc[mt][nt][r], p.rnd); continue; }
          if (p.out32) { epi32_plain(p, m, n, acc[mt][nt][r]); continue; }
          const float y = (float)(AT)(VAR ? silu_col(p.silu_cols, n, acc[mt][nt][r]) : acc[mt][nt][r]);
          if (p.epi == EPI_STORE) out[(size_t)m * p.ldo + n] = (AT)y;
          else {
            AT* h = (AT*)p.resid;
            h[(size_t)m * p.ldo + n] = (AT)((float)h[(size_t)m * p.ldo + n] + y);
          }
        }
      }
    }
  };
  if constexpr (GROUPED && !SWIGLU) store(std::false_type{});
  else if (SWIGLU ? p.glu.kind != GLU_SILU : p.silu_cols > bn * BN) store(std::true_type{});
  else store(std::false_type{});
}

// the K slices of gemm_tile_kernel, added in slice order, + the epilogue (EPI_STORE / EPI_RESID); 4 columns per thread
template <typename AT>
__global__ __launch_bounds__(256) void splitk_epilogue_kernel(GemmParams p) {
  const size_t i4 = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t total4 = (size_t)p.M * p.N / 4;
  if (i4 >= total4) return;
  const size_t e0 = i4 * 4;
  const int m = (int)(e0 / p.N), n = (int)(e0 % p.N);
  f32x4 a = {0.f, 0.f, 0.f, 0.f};
  for (int z = 0; z < p.ksplit; ++z) a += *(const f32x4*)(p.ws + (size_t)z * p.M * p.N + e0);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (p.out32) { epi32_plain(p, m, n + j, round_rt(a[j], p.rnd)); continue; }      // (p.rnd: plain stores only)
    const float y = (float)(AT)silu_col(p.silu_cols, n + j, a[j]);
    if (p.epi == EPI_STORE) ((AT*)p.out)[(size_t)m * p.ldo + n + j] = (AT)y;
    else { AT* h = (AT*)p.resid; h[(size_t)m * p.ldo + n + j] = (AT)((float)h[(size_t)m * p.ldo + n + j] + y); }
  }
}

constexpr int BM2 = 256, BN2 = 256;
template <bool SWIGLU>
__device__ __forceinline__ bool epilogue_varies(const GemmParams& p, int bn) { return SWIGLU ? p.glu.kind != GLU_SILU : p.silu_cols > bn * BN2; }

// the epilogue of the 256 x 256 tiles (2 x 4 waves, 128 x 64 per wave): lane (c16, g) holds C[m = 4g + r][n = c16] of
// every 16 x 16 tile
// VAR: another unit than silu, or a plain store with silu columns (common.h)
// (rows m4 .. m4 + 3 of the wave's 64 columns)
template <typename AT, bool SWIGLU, bool VAR, bool LOGITS = false>
__device__ __forceinline__ void tile256_epilogue_row(const GemmParams& p, const f32x4 (&acc)[4], int m4, int bn, int wn, int c16) {
  AT* out = (AT*)p.out;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
      const int m = m4 + r;
      if (m >= p.M) continue;
      if constexpr (SWIGLU) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = bn * 128 + wn * 32 + j * 16 + c16;
          if (n >= p.pair_offset) continue;
          if (p.out32) { epi32_swiglu(p, m, n, acc[j][r], acc[j + 2][r]); continue; }
          out[(size_t)m * p.ldo + n] = VAR ? (AT)glu_f(p.glu, acc[j][r], acc[j + 2][r]) : silu16<AT>(acc[j][r], acc[j + 2][r]);
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          const int n = bn * BN2 + wn * 64 + nt * 16 + c16;
          if (n >= p.N) continue;
          if constexpr (LOGITS) { ((float*)p.out)[(size_t)m * p.ldo + n] = (float)(AT)acc[nt][r]; continue; }
          if (p.out32) { epi32_plain(p, m, n, acc[nt][r]); continue; }
          const float y = (float)(AT)(VAR ? silu_col(p.silu_cols, n, acc[nt][r]) : acc[nt][r]);
          if (p.epi == EPI_STORE) out[(size_t)m * p.ldo + n] = (AT)y;
          else {
            AT* h = (AT*)p.resid;
            h[(size_t)m * p.ldo + n] = (AT)((float)h[(size_t)m * p.ldo + n] + y);
          }
        }
      }
    }
}

template <typename AT, bool SWIGLU, bool VAR, bool LOGITS = false>
__device__ __forceinline__ void tile256_epilogue(const GemmParams& p, f32x4 (&acc)[8][4], int m0, int bn, int wm, int wn, int c16, int g) {
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) tile256_epilogue_row<AT, SWIGLU, VAR, LOGITS>(p, acc[mt], m0 + wm * 128 + mt * 16 + 4 * g, bn, wn, c16);
}

// Grouped form: whole rows.  A wave's tile goes through its own strip of LDS, 64 rows at a time, and leaves it as 16-byte pieces of
// rows (out_rows may scatter them): 16 stores per wave instead of 128.  The LDS must be free (every DMA landed, every read done).
template <typename AT, bool SWIGLU, bool VAR>
__device__ __forceinline__ void tile256_epilogue_rows(const GemmParams& p, f32x4 (&acc)[8][4], unsigned char* lds, int bn, int wave, int lane, int place0) {
  constexpr int WC = SWIGLU ? 32 : 64, LDW = WC + 8, NP = WC / 8;
  const int wm = wave >> 2, wn = wave & 3, c16 = lane & 15, g = lane >> 4;
  AT* strip = (AT*)lds + (size_t)wave * 64 * LDW;
  const int n0 = bn * 4 * WC + wn * WC, cols = SWIGLU ? p.pair_offset : p.N;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        AT* row = strip + (mt * 16 + 4 * g + r) * LDW + c16;
        const f32x4 (&a)[4] = acc[hf * 4 + mt];
        if constexpr (SWIGLU) {
#pragma unroll
          for (int j = 0; j < 2; ++j) row[j * 16] = (AT)(VAR ? glu_f(p.glu, a[j][r], a[j + 2][r]) : silu_mul(a[j][r], a[j + 2][r]));
        } else {
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) row[nt * 16] = (AT)a[nt][r];
        }
      }
    asm volatile("" ::: "memory");                     // (a wave's LDS operations complete in order)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int piece = i * 64 + lane, row = piece / NP, c8 = piece % NP, m = wm * 128 + hf * 64 + row, n = n0 + c8 * 8;
      if (m >= p.M || n >= cols) continue;
      const int orow = p.out_rows != nullptr ? p.out_rows[place0 + m] : place0 + m;
      *(u32x4*)((AT*)p.out + (size_t)orow * p.ldo + n) = *(const u32x4*)(strip + row * LDW + c8 * 8);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  }
}

// The residual epilogue (h += y in place) with the loads of h batched: written as in tile256_epilogue every load of
// h sits behind the previous store to h (same array: the compiler keeps the order) -- 128 dependent round trips per
// wave, ~15 us per 256 x 256 block, 13 % of o_proj at 8 x 1024 rows.  Here the 16 values of an M tile are fetched in one
// round trip, then added and stored.
template <typename AT, typename HT>        // HT: storage of the residual stream (AT, or float in the PagedKVCache mode: h += y unrounded)
__device__ __forceinline__ void tile256_epilogue_resid(const GemmParams& p, f32x4 (&acc)[8][4], int m0, int bn, int wm, int wn, int c16, int g) {
  HT* h = (HT*)p.resid;
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    HT hv[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const int m = min(m0 + wm * 128 + mt * 16 + 4 * g + r, p.M - 1);
        const int n = min(bn * BN2 + wn * 64 + nt * 16 + c16, p.N - 1);
        hv[r][nt] = h[(size_t)m * p.ldo + n];
      }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const int m = m0 + wm * 128 + mt * 16 + 4 * g + r;
        const int n = bn * BN2 + wn * 64 + nt * 16 + c16;
        if (m >= p.M || n >= p.N) continue;
        if constexpr (std::is_same<HT, float>::value) h[(size_t)m * p.ldo + n] = hv[r][nt] + acc[mt][nt][r];
        else h[(size_t)m * p.ldo + n] = (AT)((float)hv[r][nt] + (float)(AT)acc[mt][nt][r]);
      }
  }
}

// The same epilogues through LDS: a wave writes ROWS rows of its tile to a strip of its own and takes them out as 16-byte pieces of rows -- 64 to
// 128 bytes of a row side by side where a register is one column of four rows: 2 or 4 bytes a lane, 64 to 256 stores (and loads of the residual) a
// wave, each of which takes the CU's address unit 16 cycles.  Element stores -> strips, us: 8192 rows, 6144 x 4096 318 -> 297, 28672 x 4096 SwiGLU
// 1583 -> 1542, 4096 x 14336 with the residual 705 -> 690, 2048 x 2048 64 -> 56; 4096 rows, 16384 x 2048 249 -> 213.
// Where rows are whole 16-byte pieces (host: GemmParams::strips); the LDS must be free.
template <typename ST, int WC, typename Value, typename Emit>
__device__ __forceinline__ void tile256_strips(unsigned char* lds, int wave, int lane, Value value, Emit emit) {
  constexpr int ROWS = WC * sizeof(ST) > 128 ? 32 : 64, PER = 16 / sizeof(ST), LDW = WC + PER, NP = WC / PER, MTP = ROWS / 16;
  const int c16 = lane & 15, g = lane >> 4;
  ST* strip = (ST*)lds + (size_t)wave * ROWS * LDW;
#pragma unroll
  for (int pass = 0; pass < 128 / ROWS; ++pass) {
#pragma unroll
    for (int mt = 0; mt < MTP; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ct = 0; ct < WC / 16; ++ct) strip[(mt * 16 + 4 * g + r) * LDW + ct * 16 + c16] = value(pass * MTP + mt, r, ct);
    asm volatile("" ::: "memory");                     // (a wave's LDS operations complete in order)
    __builtin_amdgcn_wave_barrier();
    u32x4 v[ROWS * NP / 64];
#pragma unroll
    for (int i = 0; i < ROWS * NP / 64; ++i) {
      const int piece = i * 64 + lane;
      v[i] = *(const u32x4*)(strip + (piece / NP) * LDW + (piece % NP) * PER);
    }
    emit(pass * ROWS, v, [&](int i) { return (i * 64 + lane) / NP; }, [&](int i) { return (i * 64 + lane) % NP * PER; });
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  }
}

// a K slice's partial tile, float32 (rows of N values, N a multiple of 16); with the elements stored one by one, us: 700 rows, 6144 x 4096 76.5, here 75.0;
// 4096 x 14336 93.0, 91.5; 4096 x 4096 43.0, 42.3
__device__ __forceinline__ void tile256_partial(const GemmParams& p, f32x4 (&acc)[8][4], unsigned char* lds, int m0, int bn, int wave, int lane) {
  float* wz = p.ws + (size_t)blockIdx.z * p.M * p.N;
  const int mw = m0 + (wave >> 2) * 128, n0 = bn * BN2 + (wave & 3) * 64;
  __syncthreads();
  tile256_strips<float, 64>(lds, wave, lane, [&](int mt, int r, int ct) { return acc[mt][ct][r]; }, [&](int row0, auto& v, auto row, auto col) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(v) / 16); ++i) {
      const int m = mw + row0 + row(i), n = n0 + col(i);
      if (m < p.M && n < p.N) *(u32x4*)(wz + (size_t)m * p.N + n) = v[i];
    }
  });
}

template <typename AT, bool SWIGLU, bool VAR, bool LOGITS = false>
__device__ __forceinline__ void tile256_epilogue_strips(const GemmParams& p, f32x4 (&acc)[8][4], unsigned char* lds, int m0, int bn, int wave, int lane) {
  constexpr int WC = SWIGLU ? 32 : 64;
  const int n0 = bn * 4 * WC + (wave & 3) * WC, cols = SWIGLU ? p.pair_offset : p.N, c16 = lane & 15;
  const int mw = m0 + (wave >> 2) * 128;
  // pieces of ST into rows of `dst`, stride ld; add: the residual
  auto store = [&](auto* dst, size_t ld, int row0, auto& v, auto row, auto col) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(v) / 16); ++i) {
      const int m = mw + row0 + row(i), n = n0 + col(i);
      if (m < p.M && n < cols) *(u32x4*)(dst + (size_t)m * ld + n) = v[i];
    }
  };
  auto fetch = [&](const auto* src, int row0, auto& h, auto row, auto col) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(h) / 16); ++i)
      h[i] = *(const u32x4*)(src + (size_t)min(mw + row0 + row(i), p.M - 1) * p.ldo + min(n0 + col(i), cols - (int)(16 / sizeof(*src))));
  };
  if constexpr (SWIGLU) {
    if (p.split_out) {                                 // two bf16 terms, hi = bf16(y), lo = bf16(y - hi): what the down projection multiplies
      tile256_strips<uint32_t, WC>(lds, wave, lane, [&](int mt, int r, int ct) {
        float y = glu32(p.glu, acc[mt][ct][r], acc[mt][ct + 2][r]);
        asm("" : "+v"(y));                               // (the product is rounded before lo takes hi off it: no FMA over both)
        const bf16 hi = (bf16)y, lo = (bf16)(y - (float)hi);
        return (uint32_t)__builtin_bit_cast(uint16_t, hi) | (uint32_t)__builtin_bit_cast(uint16_t, lo) << 16;
      }, [&](int row0, auto& v, auto row, auto col) {
#pragma unroll
        for (int i = 0; i < (int)(sizeof(v) / 16); ++i) {
          const int m = mw + row0 + row(i), n = n0 + col(i);
          if (m >= p.M || n >= cols) continue;
          uint16_t* o = (uint16_t*)p.out + (size_t)m * (2 * p.ldo) + n;
          *(uint2*)o = uint2{(v[i].x & 0xffffu) | (v[i].y << 16), (v[i].z & 0xffffu) | (v[i].w << 16)};
          *(uint2*)(o + p.ldo) = uint2{(v[i].x >> 16) | (v[i].y & 0xffff0000u), (v[i].z >> 16) | (v[i].w & 0xffff0000u)};
        }
      });
    } else if (p.out32) {
      tile256_strips<float, WC>(lds, wave, lane, [&](int mt, int r, int ct) { return glu32(p.glu, acc[mt][ct][r], acc[mt][ct + 2][r]); },
                                [&](int row0, auto& v, auto row, auto col) { store((float*)p.out, p.ldo, row0, v, row, col); });
    } else {
      tile256_strips<AT, WC>(lds, wave, lane, [&](int mt, int r, int ct) {
        return VAR ? (AT)glu_f(p.glu, acc[mt][ct][r], acc[mt][ct + 2][r]) : silu16<AT>(acc[mt][ct][r], acc[mt][ct + 2][r]);
      }, [&](int row0, auto& v, auto row, auto col) { store((AT*)p.out, p.ldo, row0, v, row, col); });
    }
  } else if (LOGITS || p.out32) {
    tile256_strips<float, WC>(lds, wave, lane, [&](int mt, int r, int ct) { return LOGITS ? (float)(AT)acc[mt][ct][r] : acc[mt][ct][r]; },
                              [&](int row0, auto& v, auto row, auto col) {
      if (LOGITS || p.epi == EPI_STORE) { store((float*)p.out, p.ldo, row0, v, row, col); return; }
      f32x4 h[sizeof(v) / 16];
      fetch((const float*)p.resid, row0, (u32x4(&)[sizeof(v) / 16])h, row, col);
#pragma unroll
      for (int i = 0; i < (int)(sizeof(v) / 16); ++i) v[i] = __builtin_bit_cast(u32x4, h[i] + __builtin_bit_cast(f32x4, v[i]));
      store((float*)p.resid, p.ldo, row0, v, row, col);
    });
  } else {
    tile256_strips<AT, WC>(lds, wave, lane, [&](int mt, int r, int ct) { return (AT)(VAR ? silu_col(p.silu_cols, n0 + ct * 16 + c16, acc[mt][ct][r]) : acc[mt][ct][r]); },
                           [&](int row0, auto& v, auto row, auto col) {
      if (p.epi == EPI_STORE) { store((AT*)p.out, p.ldo, row0, v, row, col); return; }
      u32x4 h[sizeof(v) / 16];
      fetch((const AT*)p.resid, row0, h, row, col);
#pragma unroll
      for (int i = 0; i < (int)(sizeof(v) / 16); ++i) {
        AT* y = (AT*)&v[i];
        const AT* hv = (const AT*)&h[i];
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = (AT)((float)hv[j] + (float)y[j]);
      }
      store((AT*)p.resid, p.ldo, row0, v, row, col);
    });
  }
}

// ---------------------------------------------------------------------------------------------
// 256 x 256 x 64 tile, 8 waves (2 in M x 4 in N, 128 x 64 per wave = 8 x 4 MFMA tiles), BOTH operands staged in
// LDS.  Why: with W fragments read per wave from global memory the 128 x 128 kernel moves 48 KB from L2 per
// 2.1 MFLOP (44 flop/B) and sits on the L2 -> CU bandwidth (~19 TB/s at its 840 TFLOP/s); here a K step moves
// 64 KB per 8.4 MFLOP (131 flop/B).  The W block of a K step keeps its tile-major order in LDS -- a fragment is one
// contiguous KiB, read conflict-free -- so the copy global -> registers -> LDS is a plain 16-byte lane-linear move.
// Double-buffered: the next step's 8 loads per thread are in flight during the current step's 64 MFMAs per wave.
// SWIGLU: the block covers 128 gate columns and the 128 matching up columns; a wave's four N tiles are two gate
// tiles + their up tiles.
constexpr int A2_BYTES = BM2 * LDA * 2;                 // one X image (rows padded to 144 B)
constexpr int B2_BYTES = BN2 * BK * 2;                  // one W image: 16 row tiles x 2 k blocks x 1 KiB
constexpr int LDS2_BYTES = 2 * (A2_BYTES + B2_BYTES);
constexpr int AFR = 4;                                  // A fragments in flight from LDS (ring): item i + 3 is read while item i multiplies
constexpr int SYNC_AT = 13;                             // the item in front of which the K step's barrier sits
constexpr int STORE_AT = 11;                            // the item (of 16 per K step) after which the next tile is written to LDS

// BD ("B direct", A/B variant behind MI_GEMM_B_DIRECT): the W fragments do not go through LDS -- in the tile-major
// layout a fragment is one contiguous KiB, so each wave loads the 8 fragments of its four N tiles for the NEXT K step
// straight into a second register set (two sets in turn, the K loop is unrolled by two); LDS then carries only the X
// tile (16 instead of 24 fragment reads per wave and step, half the stores).  Measured 2 % SLOWER than both operands
// in LDS (68.5 k vs 69.9 k prefill tok/s): the LDS pipe was not the limit, the instruction order was (below).
template <typename AT, bool SWIGLU, bool BD, bool LOGITS = false>
__global__ __launch_bounds__(512) void gemm_tile256_kernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem2[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;              // 2 x 4 waves
  const int c16 = lane & 15, g = lane >> 4;
  const int bm = blockIdx.x, bn = blockIdx.y;           // M fastest: co-scheduled blocks share the W tiles in L2
  const int m0 = bm * BM2;
  const int nk = p.K / BK, nkw = p.kw / BK;
  const AT* x = (const AT*)p.x;
  const int ntiles_w = p.N / 16;
  auto a_img = [&](int buf) { return (AT*)(smem2 + (size_t)buf * A2_BYTES); };
  auto b_img = [&](int buf) { return smem2 + 2 * (size_t)A2_BYTES + (size_t)buf * B2_BYTES; };

  // the 16 W row tiles of this block, in LDS order: tile slot s (0..15)
  auto w_tile_of = [&](int s) -> int {
    int t;
    if constexpr (!SWIGLU) t = (bn * BN2) / 16 + s;
    else t = (bn * 128 + (s >> 2) * 32 + (s & 1) * 16 + ((s >> 1) & 1) * p.pair_offset) / 16;   // wave wn = s>>2: gate, gate, up, up
    return min(t, ntiles_w - 1);
  };

  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- global -> registers: X 256 rows x 8 chunks = 2048 pieces, W 16 tiles x 2 k blocks x 64 lanes = 2048 pieces.
  // STRAIGHT-LINE loads (no exec mask, no branch): a load under a condition makes hipcc drain the vmcnt queue at the
  // join -- here that was an exposed L2 round trip per K step.  Rows past M read row M - 1 and are zeroed on the
  // way into LDS; the step after the last re-reads the last step.
  constexpr int NB = BD ? 1 : 4;
  u32x4 areg[4], breg[NB];
  const AT* arow[4];
  const char* brow[NB];
  bool aok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + 512 * i, row = c >> 3, kq = c & 7;
    aok[i] = m0 + row < p.M;
    arow[i] = x + (size_t)min(m0 + row, p.M - 1) * p.ldx + kq * 8;
    if constexpr (!BD) {
      const int s = c >> 7, kb = (c >> 6) & 1, l = c & 63;
      brow[i] = (const char*)p.w + ((size_t)w_tile_of(s) * (p.kw / 32) + (size_t)kb) * 1024 + l * 16;
    }
  }
  const char* bptr[4];                                   // BD: this wave's four N tiles, lane-linear
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) bptr[nt] = (const char*)p.w + (size_t)w_tile_of(wn * 4 + nt) * (p.kw / 32) * 1024 + lane * 16;
  auto load_a = [&](int ks) {
    const int ka = (ks * BK) % p.ka;
#pragma unroll
    for (int i = 0; i < 4; ++i) areg[i] = *(const u32x4*)(arow[i] + ka);
    if constexpr (!BD) {
#pragma unroll
      for (int i = 0; i < 4; ++i) breg[i] = *(const u32x4*)(brow[i] + (size_t)(ks % nkw) * 2048);
    }
  };
  auto load_bd = [&](int ks, u32x4 (&dst)[2][4]) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) dst[kb][nt] = *(const u32x4*)(bptr[nt] + (size_t)((ks % nkw) * 2 + kb) * 1024);
  };
  auto store_ab = [&](int buf) {
    AT* A = a_img(buf);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + 512 * i, row = c >> 3, kq = c & 7;
      *(u32x4*)&A[row * LDA + kq * 8] = aok[i] ? areg[i] : u32x4{0u, 0u, 0u, 0u};
    }
    if constexpr (!BD) {
      unsigned char* B = b_img(buf);
#pragma unroll
      for (int i = 0; i < 4; ++i) *(u32x4*)(B + (size_t)(tid + 512 * i) * 16) = breg[i];     // (slot, kb, lane) order = piece index
    }
  };

  u32x4 bset0[2][4], bset1[2][4];                        // BD: the W fragments of the current / the next K step
  // The fragment pipeline runs ACROSS the K steps: 16 (k block, M tile) items of 4 MFMAs per step; the A fragment of
  // item i + 3 is read from LDS while item i multiplies (ring of AFR registers; 16 % AFR == 0, so the ring index carries
  // over), and for the last three items of a step "item i + 3" is item 0..2 of the NEXT step, read from the other
  // buffer.  That buffer is complete once every wave has stored its share (after item STORE_AT) -- so the step's one
  // barrier sits in front of item SYNC_AT, not at the end of the step, and the wait for the first fragments of a
  // step hides behind the previous step's last 12 MFMAs instead of stopping every wave of the workgroup at once.
  u32x4 bf[2][4], af[AFR];
  auto a_frag = [&](const AT* A, int it) {
    return *(const u32x4*)&A[(wm * 128 + (it & 7) * 16 + c16) * LDA + (it >> 3) * 32 + g * 8];
  };
  auto b_frags = [&](const unsigned char* B, int kb, u32x4 (&dst)[4]) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) dst[nt] = *(const u32x4*)(B + (size_t)(((wn * 4 + nt) * 2 + kb) * 64 + lane) * 16);
  };
  // one K step: `bc` holds this step's W fragments (BD), `bn` receives the next step's
  auto step = [&](int ks, u32x4 (&bc)[2][4], u32x4 (&bn)[2][4]) {
    const int cur = ks & 1;
    load_a(min(ks + 1, nk - 1));
    if constexpr (BD) load_bd(min(ks + 1, nk - 1), bn);
    __builtin_amdgcn_sched_barrier(0);           // keep the loads HERE, a whole step of MFMAs ahead of their use (hipcc
                                                 // otherwise sinks them next to the LDS stores at the bottom of the step)
    const AT* A = a_img(cur);
    const AT* An = a_img(cur ^ 1);
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      if (it == SYNC_AT) {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();                         // the other buffer holds the next step's tile; this step's reads are done
        __builtin_amdgcn_sched_barrier(0);
      }
      const int nx = it + AFR - 1;
      af[nx % AFR] = nx < 16 ? a_frag(A, nx) : a_frag(An, nx - 16);
      if constexpr (!BD) {
        if (it == 3) b_frags(b_img(cur), 1, bf[1]);
        if (it == SYNC_AT) b_frags(b_img(cur ^ 1), 0, bf[0]);     // (bf[0] is dead since item 7)
      }
#if MI_GEMM_VARIANT == 1
      __builtin_amdgcn_s_setprio(1);
#endif
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        acc[it & 7][nt] = mfma16<AT>(af[it % AFR], BD ? bc[it >> 3][nt] : bf[it >> 3][nt], acc[it & 7][nt]);
#if MI_GEMM_VARIANT == 1
      __builtin_amdgcn_s_setprio(0);
#endif
      // the order is imposed on hipcc's scheduler (sched_group_barrier: 0x100 = LDS read, 0x008 = MFMA); left alone
      // it bunches the fragment reads and waits for them in front of single MFMAs
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (!BD && (it == 3 || it == SYNC_AT)) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      if (it == STORE_AT) {
        // the next step's tile goes into the other buffer (its readers finished before the last barrier): the loads
        // have had three quarters of a step to arrive
        __builtin_amdgcn_sched_barrier(0);
        store_ab(cur ^ 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  load_a(0);
  if constexpr (BD) load_bd(0, bset0);
  store_ab(0);
  __syncthreads();
  // static priority for the younger wave of every SIMD (waves 4..7 lose every issue arbitration by age otherwise):
  // prefill 72.9 k -> 73.5 k tok/s, two runs each on one box.  (Priority flipped around every MFMA group: -1 %.)
  if (wave >= 4) __builtin_amdgcn_s_setprio(1);
  if constexpr (!BD) b_frags(b_img(0), 0, bf[0]);
#pragma unroll
  for (int i = 0; i < AFR - 1; ++i) af[i] = a_frag(a_img(0), i);
  for (int ks = 0; ks < nk; ks += 2) {
    step(ks, bset0, bset1);
    if (ks + 1 < nk) step(ks + 1, bset1, bset0);
  }

  if constexpr (!SWIGLU && !LOGITS) {
    if (p.epi == EPI_RESID) {
      if (p.out32) tile256_epilogue_resid<AT, float>(p, acc, m0, bn, wm, wn, c16, g);
      else tile256_epilogue_resid<AT, AT>(p, acc, m0, bn, wm, wn, c16, g);
      return;
    }
  }
  if constexpr (LOGITS) tile256_epilogue<AT, SWIGLU, false, true>(p, acc, m0, bn, wm, wn, c16, g);
  else if (epilogue_varies<SWIGLU>(p, bn)) tile256_epilogue<AT, SWIGLU, true>(p, acc, m0, bn, wm, wn, c16, g);
  else tile256_epilogue<AT, SWIGLU, false>(p, acc, m0, bn, wm, wn, c16, g);
}


// ---------------------------------------------------------------------------------------------------------------
// 256 x 256 x 64 tile, both operands staged by LDS-DMA (global_load_lds_dwordx4): no staging registers, no ds_write, the
// copies of a K tile stay in flight across barriers for two to four phases, and the two waves of a SIMD take the matrix
// core in turn.  Same wave grid and accumulator layout as gemm_tile256_kernel (2 x 4 waves, 128 x 64 per wave,
// acc[8][4]), same MFMA chain per accumulator (so the same float32 sums, bit for bit), same epilogue.
// Mistral-7B linears over 8 x 1024 rows, random bf16 operands, interleaved rounds in one process (tools/debug/
// gemm_prefill_ab.py): 1.15 / 1.03 / 1.15 / 1.14 PFLOP/s (q|k|v, o, gate|up, down) on the register-staged tile,
// 1.38 / 1.17 / 1.35 / 1.38 here with phases of 16 MFMAs; the float32-cache prompt's products (two terms of x) 617 / 2790 us
// (q|k|v, gate|up) so, 613 / 2757 with the 32 of now.  What bounds it is power: the matrix core is busy three cycles of four at 1.6 to 1.75 GHz
// (s_memtime against the wall clock in the loop; the same clock counts 2.2 in a light kernel).
//
// LDS, all 160 KiB: three buffers of 32 KiB for A, two for B; each is two UNITS of 16 KiB -- a unit is what all 8 waves stage together
// (two 1-KiB DMA instructions per wave):
//     A-h0 / A-h1   rows {wm * 128 + h * 64 + [0, 64)} of the X tile (128 rows x 128 B), image row ir = wm * 64 + r
//     B-k0 / B-k1   the 16 W row tiles of k block kb: 16 fragments of 1 KiB in tile-major order (a fragment read is one
//                   contiguous KiB: conflict-free as it lies)
// A image: the DMA writes lane-linear (base + 16 lane), so the layout is chosen through the SOURCE address of each lane.
// Image rows are paired into 256-byte bank rows; piece (ir, q) (q = 16-byte chunk 0..7 of the row's 128 bytes) lies at
//     (ir >> 1) * 256 + ((((ir & 1) << 3) | q) ^ ((ir >> 1) & 7)) * 16
// -- every lane group of a ds_read_b128 fragment read ({0-3, 12-15, 20-27}, ... : 16 rows x one or two q) hits 16
// different 16-byte columns (checked exhaustively), and the 8 lanes that fill a row fetch its whole 128-byte line.
//
// Schedule (ping-pong).  A K tile is two phases of 32 MFMAs per wave, one per k block.  A phase is
//     [reads of ITS fragments, stage two units, s_waitcnt lgkmcnt(0), s_waitcnt vmcnt(8)] s_barrier [32 MFMAs] s_barrier;
// waves 4..7 -- the second wave of every SIMD -- enter through one extra barrier (and waves 0..3 leave through one), so
// every s_barrier pairs the end of one group's read section with the end of the other's MFMA section: while one wave of a
// SIMD reads and issues its DMA, the other has the matrix core.  Reads come BEFORE the DMA issue: an LDS-DMA instruction
// holds the wave's issue for 60..180 cycles (the CU's one address unit serves four waves at once), the fragments arrive
// meanwhile.
//   stage:  j=0: A-h0(t+2), B-k1(t+1)     j=1: A-h1(t+2), B-k0(t+2)
// Write-after-read: the reads a group issues in phase Q have completed at that group's next barrier (lgkmcnt(0)), both
// groups' two barriers after phase Q began; a unit last read in phase Q is restaged in phase Q + 1 at the earliest
// (A(t-1), whose buffer A(t+2) takes: (t-1, 1) -> (t, 0); B-k1(t-1): (t-1, 1) -> (t, 0); B-k0(t): (t, 0) -> (t, 1)).
// Read-after-write: a wave's DMA has landed when its counted vmcnt wait says so, everybody's when both groups have passed
// the barrier behind that wait -- waited for in the read section of phase W, first read in phase W + 1:
//     unit          staged in     waited for in   first read in   DMAs issued since (may stay in flight)
//     A-h0(t+2)     (t, j=0)      (t+1, j=1)      (t+2, j=0)      (in order: landed before A-h1(t+2))
//     B-k1(t+1)     (t, j=0)      (t+1, j=0)      (t+1, j=1)      4 units -> vmcnt(8)
//     A-h1(t+2), B-k0(t+2)  (t, j=1)  (t+1, j=1)  (t+2, j=0)      4 units -> vmcnt(8)
// (vmcnt counts in order, and these DMAs are the loop's only vector-memory instructions.)  Past the last tile the stages
// repeat the last tile's sources -- straight-line, the counts stay what the table says -- into units nobody reads again.
// Measured and dropped with phases of 16 MFMAs (q|k|v / down): lockstep phases with the next phase's
// fragments read one phase ahead and ONE barrier per phase 1.26 / 1.25 PFLOP/s; this ping-pong with the DMA issued in
// front of the reads 1.29 / 1.30; the DMA issued at the head of the MFMA section 1.25 / 1.24; no s_setprio: the same.
constexpr int DMA_BUF = 65536, DMA_UNIT = 16384;
constexpr int DMA256_B = 6 * DMA_UNIT, DMA256_LDS = 10 * DMA_UNIT;

__device__ __forceinline__ void dma_kib(const void* gsrc, unsigned lds_dst) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(gsrc), "s"(lds_dst) : "memory");
}
typedef __attribute__((address_space(3))) u32x4 lds_u32x4_t;

// GROUPED: as in gemm_tile_kernel
template <typename AT, bool SWIGLU, bool GROUPED = false, bool LOGITS = false>
__global__ __launch_bounds__(512) void gemm_dma256_kernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem2[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;              // 2 x 4 waves
  const int c16 = lane & 15, g = lane >> 4;
  const int bm = blockIdx.x, bn = blockIdx.y;
  int m0 = bm * BM2, place0 = 0;
  if constexpr (GROUPED) {
    if (!group_of_tile<AT, SWIGLU>(p, bm, bn * (SWIGLU ? 128 : BN2), place0)) return;
    m0 = 0;
  }
  // K split over gridDim.z workgroups (a prompt of 256..4095 rows against N = 4096: the (M, N) grid alone leaves most CUs
  // idle): slice z multiplies the K tiles [tb, tb + nk) and leaves its float32 partial tile in ws[z][M][N];
  // splitk_epilogue_kernel adds the slices in order and applies the epilogue (host: >= 2 tiles per slice)
  const int nk_all = p.K / BK, nkw = p.kw / BK;
  const int tb = (int)(((long)blockIdx.z * nk_all) / gridDim.z);
  const int nk = (int)(((long)(blockIdx.z + 1) * nk_all) / gridDim.z) - tb;
  const int ntiles_w = p.N / 16;
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem2;

  auto w_tile_of = [&](int s) -> int {                   // the 16 W row tiles of this block, in LDS order (slot s)
    int t;
    if constexpr (!SWIGLU) t = (bn * BN2) / 16 + s;
    else t = (bn * 128 + (s >> 2) * 32 + (s & 1) * 16 + ((s >> 1) & 1) * p.pair_offset) / 16;   // wave wn = s>>2: gate, gate, up, up
    return min(t, ntiles_w - 1);
  };

  // ---- DMA sources.  A unit h, instruction i (0 / 1) of this wave = image rows (2 wave + i) * 8 + [0, 8) of the unit:
  // lane -> bank row R = lane >> 4 of the instruction's four, column col = lane & 15; row in pair = col >> 3, and the
  // chunk q it must fetch so that the linear write realises the swizzle: q = (col & 7) ^ (R & 7), R & 7 = 4 i + (lane >> 4).
  const char* asrc[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rl = lane >> 4, col = lane & 15;
      const int ir = (2 * wave + i) * 8 + 2 * rl + (col >> 3);            // image row of the unit: wm' * 64 + r
      const int q = (col & 7) ^ (4 * i + rl);
      const int row = (ir >> 6) * 128 + h * 64 + (ir & 63);                 // row of the 256-row tile
      int xr = min(m0 + row, p.M - 1);
      if constexpr (GROUPED) { xr += place0; if (p.x_rows != nullptr) xr = p.x_rows[xr]; }
      asrc[h][i] = (const char*)p.x + ((size_t)xr * p.ldx + q * 8) * sizeof(AT);
    }
  const char* bsrc[2];                                                     // B unit: fragment slots 2 wave, 2 wave + 1
#pragma unroll
  for (int i = 0; i < 2; ++i) bsrc[i] = (const char*)p.w + (size_t)w_tile_of(2 * wave + i) * (p.kw / 32) * 1024 + lane * 16;

  // unit A-h / B-kb of tile t (sources past the last tile repeat it) -> the 16 KiB at LDS byte offset `off`
  auto stage_a_at = [&](int t, int h, unsigned off) {
    const int ts = tb + min(t, nk - 1);
    const size_t koff = (size_t)((ts * BK) % p.ka) * sizeof(AT);
    const unsigned dst = lds0 + off + wave * 2048;
    dma_kib(asrc[h][0] + koff, dst);
    dma_kib(asrc[h][1] + koff, dst + 1024);
  };
  auto stage_b_at = [&](int t, int kb, unsigned off) {
    const int ts = tb + min(t, nk - 1);
    const size_t koff = (size_t)((ts % nkw) * 2 + kb) * 1024;
    const unsigned dst = lds0 + off + wave * 2048;
    dma_kib(bsrc[0] + koff, dst);
    dma_kib(bsrc[1] + koff, dst + 1024);
  };
  // ---- fragment reads.  A (kb, mt4) of the unit at `off`: image row wm * 64 + mt4 * 16 + c16, chunk kb * 4 + g
  const unsigned a_lane = lds0 + (unsigned)((wm * 32 + (c16 >> 1)) * 256 + (((((c16 & 1) << 3) | g) ^ (c16 >> 1)) * 16));
  const unsigned b_lane = lds0 + (unsigned)(wn * 4 * 1024 + lane * 16);
  auto a_frags_at = [&](unsigned off, int kb, u32x4 (&dst)[4]) {
    const unsigned base = (a_lane ^ (unsigned)(kb << 6)) + off;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) dst[mt] = *(const lds_u32x4_t*)(size_t)(base + mt * 8 * 256);
  };
  auto b_frags_at = [&](unsigned off, u32x4 (&dst)[4]) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) dst[nt] = *(const lds_u32x4_t*)(size_t)(b_lane + off + nt * 1024);
  };
  // A of tile t in buffer t mod 3 = [A-h0][A-h1], B behind them in buffer t & 1 = [B-k0][B-k1]
  auto stage_b = [&](int t, int kb) { stage_b_at(t, kb, DMA256_B + (t & 1) * (2 * DMA_UNIT) + kb * DMA_UNIT); };
  auto b_frags = [&](int t, int kb, u32x4 (&dst)[4]) { b_frags_at(DMA256_B + (t & 1) * (2 * DMA_UNIT) + kb * DMA_UNIT, dst); };

  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 af[2][4], bf[4];

  auto mma = [&](int h, const u32x4 (&a)[4], const u32x4 (&b)[4]) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) acc[h * 4 + mt][nt] = mfma16<AT>(a[mt], b[nt], acc[h * 4 + mt][nt]);
  };

  {
    // prologue: tile 0 and what the phases of tiles -2 / -1 would have staged, in their order
    stage_a_at(0, 0, 0); stage_a_at(0, 1, DMA_UNIT); stage_b(0, 0);
    stage_a_at(1, 0, 2 * DMA_UNIT); stage_b(0, 1); stage_a_at(1, 1, 3 * DMA_UNIT); stage_b(1, 0);
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    if (wave >= 4) asm volatile("s_barrier" ::: "memory");
#define PP_READS_DONE(VM) do { __builtin_amdgcn_sched_barrier(0); asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); \
      if (VM >= 0) asm volatile("s_waitcnt vmcnt(%0)" :: "i"(VM < 0 ? 0 : VM) : "memory"); \
      asm volatile("s_barrier" ::: "memory"); __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_setprio(1); } while (0)
#define PP_MMA_DONE() do { __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_setprio(0); asm volatile("s_barrier" ::: "memory"); \
      __builtin_amdgcn_sched_barrier(0); } while (0)
#define PP_ORDER() __builtin_amdgcn_sched_barrier(0)
    unsigned ra = 0, sa = 4 * DMA_UNIT;                            // A of tile t, of tile t + 2
    for (int t = 0; t < nk; ++t) {
      b_frags(t, 0, bf); a_frags_at(ra, 0, af[0]); a_frags_at(ra + DMA_UNIT, 0, af[1]); PP_ORDER();
      stage_a_at(t + 2, 0, sa); stage_b(t + 1, 1);
      PP_READS_DONE(8);
      mma(0, af[0], bf); mma(1, af[1], bf);
      PP_MMA_DONE();
      b_frags(t, 1, bf); a_frags_at(ra, 1, af[0]); a_frags_at(ra + DMA_UNIT, 1, af[1]); PP_ORDER();
      stage_a_at(t + 2, 1, sa + DMA_UNIT); stage_b(t + 2, 0);
      PP_READS_DONE(8);
      mma(0, af[0], bf); mma(1, af[1], bf);
      PP_MMA_DONE();
      ra = ra == 4 * DMA_UNIT ? 0 : ra + 2 * DMA_UNIT;
      sa = sa == 4 * DMA_UNIT ? 0 : sa + 2 * DMA_UNIT;
    }
#undef PP_ORDER
#undef PP_READS_DONE
#undef PP_MMA_DONE
    if (wave < 4) asm volatile("s_barrier" ::: "memory");
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // no DMA of this workgroup may land after it has left the CU

  if constexpr (!SWIGLU) {
    if (gridDim.z > 1) { tile256_partial(p, acc, smem2, m0, bn, wave, lane); return; }
  }
  if constexpr (!GROUPED) {
    if (p.strips) {
      __syncthreads();
      if (!LOGITS && epilogue_varies<SWIGLU>(p, bn)) tile256_epilogue_strips<AT, SWIGLU, true, LOGITS>(p, acc, smem2, m0, bn, wave, lane);
      else tile256_epilogue_strips<AT, SWIGLU, false, LOGITS>(p, acc, smem2, m0, bn, wave, lane);
      return;
    }
  }
  if constexpr (!SWIGLU && !LOGITS) {
    if (p.epi == EPI_RESID) {
      if (p.out32) tile256_epilogue_resid<AT, float>(p, acc, m0, bn, wm, wn, c16, g);
      else tile256_epilogue_resid<AT, AT>(p, acc, m0, bn, wm, wn, c16, g);
      return;
    }
  }
  if constexpr (GROUPED) {
    __syncthreads();
    if (SWIGLU && p.glu.kind != GLU_SILU) tile256_epilogue_rows<AT, SWIGLU, SWIGLU>(p, acc, smem2, bn, wave, lane, place0);
    else tile256_epilogue_rows<AT, SWIGLU, false>(p, acc, smem2, bn, wave, lane, place0);
  } else if constexpr (LOGITS) tile256_epilogue<AT, SWIGLU, false, true>(p, acc, m0, bn, wm, wn, c16, g);
  else if (epilogue_varies<SWIGLU>(p, bn)) tile256_epilogue<AT, SWIGLU, true>(p, acc, m0, bn, wm, wn, c16, g);
  else tile256_epilogue<AT, SWIGLU, false>(p, acc, m0, bn, wm, wn, c16, g);
}


// ---------------------------------------------------------------------------------------------------------------
// Quantised weights (w = s q + b per group of 64 k): the 256 x 256 x 64 tile on the CODES.  A K tile is one group, so
//     y[m][n] = sum_g s[n][g] (sum_k (q - c) x) + sum_g (b + c s)[n][g] (sum_k x),     c = 8 or 128, the middle of the codes,
// the inner sums as MFMAs on q - c as 16-bit integers (exact: 4 or 8 bits in the 8 of bf16), one FMA per accumulator and group, and the
// second term as a matrix product of its own: the group sums of x and b + c s in bf16 terms (hi + mid + lo = the float32 value), the six
// products of the terms above 2^-24 of the whole, 6 K / 64 columns.
// Why: the [hi | lo] copy that the dense tile takes doubles the products and the bytes of the copy.  The codes carry no rounding at all;
// [hi | lo] drops what lies below 2^-17 of a weight.  Around their middle: codes of 0..15 (255) make sums of twice the size and more that
// the biases take back; the float32 result is then 4.5e-7 from the 64-bit one (6144 x 4096, 1024 rows, 2-norm), here 1.4e-7, [hi | lo] 4.1e-7.
// Float32 rows: the largest last -- x's lo, mid and hi, then the bias columns, their smallest parts first --, so that few roundings are of the size of the
// result (16-bit rows are rounded to 16 bits behind all of this, and take the biases, largest parts first, in front: recorded greedy sequences have ties there): 1024
// x 8192, 64 float32 rows, groups of int4 whose means are 0 / 4 / 12 of their deviations, 1.6e-7 / 0.9e-7 / 0.8e-7; the biases and the hi parts in front 1.8e-7 /
// 2.4e-7 / 2.3e-7; the streaming kernel 9.7e-7 / 2.7e-7 / 1.5e-7.
// Registers: 128 accumulators + the group's sums.  A phase is two row tiles x both k blocks, so those are 32 (a quarter tile) and not
// 64.  All FMAs sit behind MFMAs, two each: those of a phase's first row tile behind the MFMAs of its second, those of its second behind the
// first MFMAs of the next phase.
// Tile, LDS images, wave grid, ping-pong and epilogues: gemm_dma256_kernel.  What differs in the schedule, all reads in read sections: phase 0 reads B-k1 and
// the scales of its own K tile (256 B of a wave's own, one dword per lane and tile), phases 0 and 1 a half of A-h0 each, 2 and 3 of A-h1, and, for the NEXT K
// tile, 2 and 3 a half of B-k0 each (into the other of two register sets).
//   stage:  j=0: A-h1(t+1)   j=1: B-k0(t+2)   j=2: B-k1(t+2)   j=3: scales(t+2), A-h0(t+2)        2 + 2 + 2 + 3 DMAs of a wave (tail: no scales, 8)
//     unit                        over a unit last read in   staged in     waited for in   first read in   DMAs issued behind it by then
//     A-h1(t+1)                   (t-1, j=3)                 (t, j=0)      (t+1, j=1)      (t+1, j=2)      2 + 2 + 3 + 2 + 2 = 11
//     B-k0(t+2)                   (t-1, j=3)                 (t, j=1)      (t+1, j=1)      (t+1, j=2)      2 + 3 + 2 + 2     = 9
//     B-k1(t+2)                   (t, j=0)                   (t, j=2)      (t+1, j=3)      (t+2, j=0)      3 + 2 + 2 + 2 + 3 = 12
//     scales(t+2), A-h0(t+2)      (t, j=0), (t, j=1)         (t, j=3)      (t+1, j=3)      (t+2, j=0)      2 + 2 + 2 + 3     = 9
// Both waits are vmcnt(9) (tail: 8), behind the phase's own staging: at j=1 B-k0 sets the number (with A-h1's 11 it would be read before it has landed), at j=3
// the scales and A-h0 do.  A unit's last readers have their data before the barrier that its next stager passes first.
constexpr int CODES_LDS = 2 * DMA_BUF + 8 * 2 * 256;

__device__ __forceinline__ void dma_kib_off(const void* base, uint32_t off, unsigned lds_dst) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(off), "s"(base), "s"(lds_dst) : "memory");
}
__device__ __forceinline__ void dma_dword_off(const void* base, uint32_t off, unsigned lds_dst) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(off), "s"(base), "s"(lds_dst) : "memory");
}
typedef __attribute__((address_space(3))) f32x4 lds_f32x4_t;

template <typename AT, bool SWIGLU, bool LOGITS, bool X3>
__global__ __launch_bounds__(512) void gemm_codes256_kernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem2[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int c16 = lane & 15, g = lane >> 4;
  int bm = blockIdx.x, bn = blockIdx.y, z = blockIdx.z, nz = gridDim.z;
  if (p.mb > 0) {                                               // (uniform) K slices of the last tiles alone
    int tile = blockIdx.x;
    z = 0; nz = 1;
    if (tile >= p.tail) { const int u = tile - p.tail; nz = p.ksplit; tile = p.tail + u / nz; z = u - u / nz * nz; }
    bn = tile / p.mb; bm = tile - bn * p.mb;
    bm = __builtin_amdgcn_readfirstlane(bm); bn = __builtin_amdgcn_readfirstlane(bn); z = __builtin_amdgcn_readfirstlane(z); nz = __builtin_amdgcn_readfirstlane(nz);
  }
  const int m0 = bm * BM2;
  // K tiles: [0, nkm) = the groups of x's terms in turn, the last term first (W is walked once per term), [nkm, nk_all) = the bias columns
  const int nkm = p.ka / BK, nk_all = nkm + p.kb / BK;
  // this workgroup's: [tb, te) (divisions run on vector registers: back to scalar ones, the DMA bases are built of them)
  const int tb = __builtin_amdgcn_readfirstlane((int)((z * (unsigned)nk_all) / nz));
  const int te = __builtin_amdgcn_readfirstlane((int)(((z + 1) * (unsigned)nk_all) / nz));
  const int ntiles_w = p.N / 16;
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem2;

  auto w_tile_of = [&](int s) -> int {
    int t;
    if constexpr (!SWIGLU) t = (bn * BN2) / 16 + s;
    else t = (bn * 128 + (s >> 2) * 32 + (s & 1) * 16 + ((s >> 1) & 1) * p.pair_offset) / 16;
    return min(t, ntiles_w - 1);
  };

  // ---- DMA sources: a base in scalar registers + 32-bit offsets of the lanes (the host checks the sizes).  A unit h, instruction i of this wave
  // = image rows (2 wave + i) * 8 + [0, 8)
  uint32_t aoff[2][2];
  const char *ga, *gb[2], *gs;                                   // of the run's first K tile: x (or the group sums), this wave's two W tiles, the scales
  int last;                                                      // the run's last K tile
  auto sources = [&](const void* x, uint32_t row_bytes, const void* w, size_t tile_bytes) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int rl = lane >> 4, col = lane & 15, ir = (2 * wave + i) * 8 + 2 * rl + (col >> 3);
        aoff[h][i] = (uint32_t)min(m0 + (ir >> 6) * 128 + h * 64 + (ir & 63), p.M - 1) * row_bytes + (uint32_t)(((col & 7) ^ (4 * i + rl)) * 16);
      }
    ga = (const char*)x;
#pragma unroll
    for (int i = 0; i < 2; ++i) gb[i] = (const char*)w + w_tile_of(2 * wave + i) * tile_bytes;
    // (in scalar registers before the loop: a pending load of a kernel argument makes the compiler wait for every LDS read with it)
    asm volatile("" : "+s"(ga), "+s"(gb[0]), "+s"(gb[1]), "+s"(gs));
  };
  const uint32_t lane16 = (uint32_t)lane * 16;
  const uint32_t soff = (uint32_t)(w_tile_of(wn * 4 + (lane & 3)) * p.G * 64 + (lane >> 2) * 4);
  const unsigned sc_lds = lds0 + 2 * DMA_BUF + wave * 512;
  auto stage_a = [&](int t, int h) {
    const char* base = ga + (size_t)((uint32_t)min(t, last) * (BK * 2));
    const unsigned dst = lds0 + (t & 1) * DMA_BUF + h * DMA_UNIT + wave * 2048;
    dma_kib_off(base, aoff[h][0], dst);
    dma_kib_off(base, aoff[h][1], dst + 1024);
  };
  auto stage_b = [&](int t, int kb) {
    const size_t koff = (uint32_t)min(t, last) * 2048 + kb * 1024;
    const unsigned dst = lds0 + (t & 1) * DMA_BUF + (2 + kb) * DMA_UNIT + wave * 2048;
    dma_kib_off(gb[0] + koff, lane16, dst);
    dma_kib_off(gb[1] + koff, lane16, dst + 1024);
  };
  auto stage_s = [&](int t) { dma_dword_off(gs + (size_t)((uint32_t)min(t, last) * 64), soff, sc_lds + (t & 1) * 256); };
  const unsigned a_lane = lds0 + (unsigned)((wm * 32 + (c16 >> 1)) * 256 + (((((c16 & 1) << 3) | g) ^ (c16 >> 1)) * 16));
  const unsigned b_lane = lds0 + (unsigned)(wn * 4 * 1024 + lane * 16);
  u32x4 af[2][2], b0[2][4], b1[4];                               // [row tile of the phase][k block]; [K tile & 1][column tile]; [column tile]
  auto a_frags = [&](int t, int j) {
    const unsigned off = (t & 1) * DMA_BUF + (j >> 1) * DMA_UNIT + (j & 1) * 2 * 8 * 256;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 2; ++i) af[i][kb] = *(const lds_u32x4_t*)(size_t)((a_lane ^ (unsigned)(kb << 6)) + off + i * 8 * 256);
  };
  auto b_frag = [&](int t, int kb, int nt) { return *(const lds_u32x4_t*)(size_t)(b_lane + (t & 1) * DMA_BUF + (2 + kb) * DMA_UNIT + nt * 1024); };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[8][4], tmp[2][4], sc = zero;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) tmp[i][j] = zero;
  auto fold2 = [&](int mt, int nt, int half) {
#pragma unroll
    for (int r = 2 * half; r < 2 * half + 2; ++r) acc[mt][nt][r] = fmaf(sc[nt], tmp[mt & 1][nt][r], acc[mt][nt][r]);
    asm volatile("" : "+v"(acc[mt][nt]));                        // (here: hipcc sinks the FMAs behind the barriers and holds the sums of several phases)
  };
  auto fold = [&](int mt) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) { fold2(mt, nt, 0); fold2(mt, nt, 1); }
  };

  // (lgkmcnt(0) as the builtin: the compiler's own count then knows that the fragments are here, and waits for B-k1 alone)
#define PP_READS_DONE(VM) do { __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_waitcnt(0xC07F); \
      if (VM >= 0) asm volatile("s_waitcnt vmcnt(%0)" :: "i"(VM < 0 ? 0 : VM) : "memory"); \
      asm volatile("s_barrier" ::: "memory"); __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_setprio(1); } while (0)
#define PP_MMA_DONE() do { __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_setprio(0); asm volatile("s_barrier" ::: "memory"); \
      __builtin_amdgcn_sched_barrier(0); } while (0)
#define PP_ORDER() __builtin_amdgcn_sched_barrier(0)
  auto phase = [&](int t, auto jt, auto pt, auto tail) __attribute__((always_inline)) {
    constexpr int J = decltype(jt)::value, P = decltype(pt)::value;
    constexpr bool TAIL = decltype(tail)::value;
    f32x4 sn;
    if constexpr (J == 0) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) b1[nt] = b_frag(t, 1, nt);
      if constexpr (!TAIL) sn = *(const lds_f32x4_t*)(size_t)(sc_lds + (t & 1) * 256 + c16 * 16);
    }
    a_frags(t, J);
    if constexpr (J >= 2) {
#pragma unroll
      for (int nt = 2 * J - 4; nt < 2 * J - 2; ++nt) b0[P ^ 1][nt] = b_frag(t + 1, 0, nt);
    }
    PP_ORDER();
    if constexpr (J == 0) stage_a(t + 1, 1);
    if constexpr (J == 1) stage_b(t + 2, 0);
    if constexpr (J == 2) stage_b(t + 2, 1);
    if constexpr (J == 3) { if constexpr (!TAIL) stage_s(t + 2); stage_a(t + 2, 0); }
    PP_READS_DONE((J & 1 ? (TAIL ? 8 : 9) : -1));
    if constexpr (TAIL) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) acc[2 * J + i][nt] = mfma16<bf16>(af[i][kb], kb ? b1[nt] : b0[P][nt], acc[2 * J + i][nt]);
    } else {
      // two FMAs behind every MFMA (16 cycles = four issues): first the last phase's second row tile (phase 0: the last K tile's), then
      // this phase's first
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        tmp[0][i & 3] = i < 4 ? mfma16<AT>(af[0][0], b0[P][i], zero) : mfma16<AT>(af[0][1], b1[i & 3], tmp[0][i & 3]);
        fold2((2 * J + 7) & 7, i >> 1, i & 1);
        PP_ORDER();
      }
      if constexpr (J == 0) sc = sn;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        tmp[1][i & 3] = i < 4 ? mfma16<AT>(af[1][0], b0[P][i], zero) : mfma16<AT>(af[1][1], b1[i & 3], tmp[1][i & 3]);
        fold2(2 * J, i >> 1, i & 1);
        PP_ORDER();
      }
    }
    PP_MMA_DONE();
  };
  auto ktile = [&](int t, auto pt, auto tail) __attribute__((always_inline)) {
    phase(t, std::integral_constant<int, 0>{}, pt, tail);
    phase(t, std::integral_constant<int, 1>{}, pt, tail);
    phase(t, std::integral_constant<int, 2>{}, pt, tail);
    phase(t, std::integral_constant<int, 3>{}, pt, tail);
  };
  // one run over n K tiles of the present sources, from an empty pipeline to an empty one
  auto run = [&](int n, auto tail) __attribute__((always_inline)) {
    constexpr bool TAIL = decltype(tail)::value;
    const std::integral_constant<int, 0> even{};
    const std::integral_constant<int, 1> odd{};
    last = n - 1;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      stage_b(t, 0); stage_b(t, 1);
      if constexpr (!TAIL) stage_s(t);
      stage_a(t, 0);
      if (t == 0) stage_a(0, 1);
    }
    asm volatile("s_waitcnt vmcnt(%0)" :: "i"(TAIL ? 8 : 9) : "memory");
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) b0[0][nt] = b_frag(0, 0, nt);
    if (wave >= 4) asm volatile("s_barrier" ::: "memory");
    int t = 0;
    for (; t + 1 < n; t += 2) {
      ktile(t, even, tail);
      ktile(t + 1, odd, tail);
    }
    if (t < n) ktile(t, even, tail);
    if (wave < 4) asm volatile("s_barrier" ::: "memory");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA of this workgroup may land in the next run's units, or after it has left the CU
    asm volatile("s_barrier" ::: "memory");
  };
  const uint32_t xrow = (uint32_t)(p.ldx * 2);
  auto groups = [&]() __attribute__((always_inline)) {                    // a run per term of x, the last one (the smallest) first
    for (int t0 = 0; t0 < nkm; t0 += p.G) {
      const int lo = max(tb, t0), hi = min(te, t0 + p.G);
      if (lo >= hi) continue;
      gs = (const char*)p.sc + (size_t)(lo - t0) * 64;
      sources((const char*)p.x + (size_t)(nkm - p.G - 2 * t0 + lo) * (BK * 2), xrow, (const char*)p.w + (size_t)(lo - t0) * 2048, (size_t)p.kw * 32);
      run(hi - lo, std::false_type{});
    }
    fold(7);
  };
  if constexpr (X3) groups();
  if (te > nkm) {                                                  // the bias columns
    const int lo = max(tb, nkm) - nkm;
    gs = nullptr;
    sources((const char*)p.xs + (size_t)lo * (BK * 2), (uint32_t)(p.kb * 2), (const char*)p.wb + (size_t)lo * 2048, (size_t)p.kb * 32);
    run(te - nkm - lo, std::true_type{});
  }
  if constexpr (!X3) groups();
#undef PP_ORDER
#undef PP_READS_DONE
#undef PP_MMA_DONE

  if constexpr (!SWIGLU) {
    if (gridDim.z > 1) { tile256_partial(p, acc, smem2, m0, bn, wave, lane); return; }
  }
  if (nz > 1) {                                                  // (whole KiB, in the registers' order)
    f32x4* dst = (f32x4*)p.ws + (((size_t)(bn * p.mb + bm - p.tail) * nz + z) * 8 + wave) * (32 * 64) + lane;
#pragma unroll
    for (int i = 0; i < 32; ++i) dst[i * 64] = acc[i >> 2][i & 3];
    return;
  }
  // (one gated unit, no silu columns: codes_fits; rows that are no whole pieces are none of the engine's)
  if (p.strips) {
    __syncthreads();
    tile256_epilogue_strips<AT, SWIGLU, false, LOGITS>(p, acc, smem2, m0, bn, wave, lane);
  } else {
    tile256_epilogue<AT, SWIGLU, false, LOGITS>(p, acc, m0, bn, wm, wn, c16, g);
  }
}

// The K slices of the kernel above, added in order, and its epilogues: a workgroup per tile and row tile of its waves
template <typename AT, bool SWIGLU, bool LOGITS>
__global__ __launch_bounds__(512) void tail_reduce_kernel(GemmParams p) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tile = blockIdx.x, mt = blockIdx.y;
  const int bn = (p.tail + tile) / p.mb, bm = (p.tail + tile) % p.mb, m4 = bm * BM2 + (wave >> 2) * 128 + mt * 16 + 4 * (lane >> 4);
  if (bm * BM2 + (wave >> 2) * 128 + mt * 16 >= p.M) return;
  const f32x4* src = (const f32x4*)p.ws + ((size_t)tile * p.ksplit * 8 + wave) * (32 * 64) + mt * 4 * 64 + lane;
  f32x4 a[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) a[nt] = src[nt * 64];
#pragma unroll 2
  for (int z = 1; z < p.ksplit; ++z)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) a[nt] += src[(size_t)z * (8 * 32 * 64) + nt * 64];
  tile256_epilogue_row<AT, SWIGLU, false, LOGITS>(p, a, m4, bn, wave & 3, lane & 15);
}

// The group sums of x for the kernel above: row m -> `parts` terms of G columns each (kernels.h: codes16_sum_part; hi + mid + lo = the float32 sum
// of the group's 64 values over x's `terms` of K columns), zeros up to kb.  One workgroup per row.  (A norm in front makes them on its way:
// rmsnorm_row_block_kernel.)
__device__ __forceinline__ void store_group_sums(const float* gsum, int G, uint16_t* xs_row, int kb, int big_first) {
  for (int c = threadIdx.x; c < kb; c += 256) {
    const int term = c / G, grp = c - term * G;
    const float v = term < CODES16_TERMS ? bf16_part(gsum[grp], codes16_sum_part(big_first ? CODES16_TERMS - 1 - term : term)) : 0.f;
    xs_row[c] = __builtin_bit_cast(uint16_t, (bf16)v);
  }
}

template <typename AT>
__global__ __launch_bounds__(256) void group_sums_kernel(const AT* x, int ldx, int terms, int K, uint16_t* xs, int kb, int big_first) {
  extern __shared__ float gsum[];
  const int row = blockIdx.x, tid = threadIdx.x, G = K / 64;
  const AT* xr = x + (size_t)row * ldx;
  for (int k = tid * 8; k < K; k += 2048) {
    float s = 0.f;
    for (int t = terms - 1; t >= 0; --t) {                       // (the smallest terms first)
      const u32x4 v = *(const u32x4*)(xr + (size_t)t * K + k);
      const AT* e = (const AT*)&v;
#pragma unroll
      for (int j = 0; j < 8; ++j) s += (float)e[j];
    }
    s = lane8_sum(s);
    if ((tid & 7) == 0) gsum[k >> 6] = s;
  }
  __syncthreads();
  store_group_sums(gsum, G, xs + (size_t)row * kb, kb, big_first);
}


// ---------------------------------------------------------------------------------------------------------------
// The same 256 x 256 x 64 tile on v_mfma_f32_32x32x16: per wave and K step 32 MFMAs of 32 cycles instead of 64 of 16.
// Why: a 16x16x32 MFMA leaves 8 of its 16 cycles for other instructions to issue, the loop has ~135 of them per 64 MFMAs
// (24 LDS reads, 8 + 8 staging loads / stores, ~45 address VALU, the waits) -- more than one wave's MFMA shadow holds;
// a 32x32x16 MFMA leaves 24 of 32 cycles, i.e. 6 issue slots per MFMA and ~190 per K step.  Same staging, same LDS images
// (the A fragment of 32 rows x 16 k reads rows at the padded 144-byte stride: the 16 lanes of a read group hit 16
// distinct 16-byte slots; the B fragment of 32 W rows x 16 k is two 256-byte runs of the tile-major image, 2 KiB apart:
// conflict-free), same barrier placement.  Item (ks16, mt) = 2 MFMAs (the wave's two 32-column N tiles); SwiGLU: N tile 0
// is the gate tile, N tile 1 the matching up tile.
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename T>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (std::is_same<T, bf16>::value)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

#ifdef MI_GEMM_M32_BUILD      // a debug build target (hipcc -DMI_GEMM_M32_BUILD, run with MI_GEMM_M32=1): measured 7 % slower than the 16 x 16 x 32 form, not in the shipped library
template <typename AT, bool SWIGLU>
__global__ __launch_bounds__(512) void gemm_tile256_m32_kernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem2[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;              // 2 x 4 waves
  const int c32 = lane & 31, h2 = lane >> 5;
  const int bm = blockIdx.x, bn = blockIdx.y;
  const int m0 = bm * BM2;
  const int nk = p.K / BK, nkw = p.kw / BK;
  const AT* x = (const AT*)p.x;
  const int ntiles_w = p.N / 16;
  auto a_img = [&](int buf) { return (AT*)(smem2 + (size_t)buf * A2_BYTES); };
  auto b_img = [&](int buf) { return smem2 + 2 * (size_t)A2_BYTES + (size_t)buf * B2_BYTES; };
  auto w_tile_of = [&](int s) -> int {
    int t;
    if constexpr (!SWIGLU) t = (bn * BN2) / 16 + s;
    else t = (bn * 128 + (s >> 2) * 32 + (s & 1) * 16 + ((s >> 1) & 1) * p.pair_offset) / 16;
    return min(t, ntiles_w - 1);
  };

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  u32x4 areg[4], breg[4];
  const AT* arow[4];
  const char* brow[4];
  bool aok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + 512 * i, row = c >> 3, kq = c & 7;
    aok[i] = m0 + row < p.M;
    arow[i] = x + (size_t)min(m0 + row, p.M - 1) * p.ldx + kq * 8;
    const int s = c >> 7, kb = (c >> 6) & 1, l = c & 63;
    brow[i] = (const char*)p.w + ((size_t)w_tile_of(s) * (p.kw / 32) + (size_t)kb) * 1024 + l * 16;
  }
  auto load_ab = [&](int ks) {
    const int ka = (ks * BK) % p.ka;
#pragma unroll
    for (int i = 0; i < 4; ++i) areg[i] = *(const u32x4*)(arow[i] + ka);
#pragma unroll
    for (int i = 0; i < 4; ++i) breg[i] = *(const u32x4*)(brow[i] + (size_t)(ks % nkw) * 2048);
  };
  auto store_ab = [&](int buf) {
    AT* A = a_img(buf);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + 512 * i, row = c >> 3, kq = c & 7;
      *(u32x4*)&A[row * LDA + kq * 8] = aok[i] ? areg[i] : u32x4{0u, 0u, 0u, 0u};
    }
    unsigned char* B = b_img(buf);
#pragma unroll
    for (int i = 0; i < 4; ++i) *(u32x4*)(B + (size_t)(tid + 512 * i) * 16) = breg[i];
  };

  // item it = (ks16 = it >> 2, mt = it & 3): A fragment of rows wm*128 + 32 mt + c32, k = 16 ks16 + 8 h2
  u32x4 af[AFR], bf[4][2];
  auto a_frag = [&](const AT* A, int it) {
    return *(const u32x4*)&A[(wm * 128 + (it & 3) * 32 + c32) * LDA + (it >> 2) * 16 + h2 * 8];
  };
  auto b_frags = [&](const unsigned char* B, int ks16, u32x4 (&dst)[2]) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int slot = wn * 4 + nt * 2 + (c32 >> 4);
      dst[nt] = *(const u32x4*)(B + (size_t)(((slot * 2 + (ks16 >> 1)) * 64) + (2 * (ks16 & 1) + h2) * 16 + (c32 & 15)) * 16);
    }
  };
  auto step = [&](int ks) {
    const int cur = ks & 1;
    load_ab(min(ks + 1, nk - 1));
    __builtin_amdgcn_sched_barrier(0);
    const AT* A = a_img(cur);
    const AT* An = a_img(cur ^ 1);
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      if (it == SYNC_AT) {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
      }
      const int nx = it + AFR - 1;
      af[nx % AFR] = nx < 16 ? a_frag(A, nx) : a_frag(An, nx - 16);
      if (it == 1) b_frags(b_img(cur), 1, bf[1]);
      if (it == 5) b_frags(b_img(cur), 2, bf[2]);
      if (it == 9) b_frags(b_img(cur), 3, bf[3]);
      if (it == SYNC_AT) b_frags(b_img(cur ^ 1), 0, bf[0]);        // (bf[0] is dead since item 3)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) acc[it & 3][nt] = mfma32<AT>(af[it % AFR], bf[it >> 2][nt], acc[it & 3][nt]);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (it == 1 || it == 5 || it == 9 || it == SYNC_AT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      if (it == STORE_AT) {
        __builtin_amdgcn_sched_barrier(0);
        store_ab(cur ^ 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  load_ab(0);
  store_ab(0);
  __syncthreads();
  b_frags(b_img(0), 0, bf[0]);
#pragma unroll
  for (int i = 0; i < AFR - 1; ++i) af[i] = a_frag(a_img(0), i);
  for (int ks = 0; ks < nk; ++ks) step(ks);

  // ---- epilogue: lane (c32, h2), register r holds C[m = (r & 3) + 8 (r >> 2) + 4 h2][n = c32] of every 32 x 32 tile
  AT* out = (AT*)p.out;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + wm * 128 + mt * 32 + (r & 3) + 8 * (r >> 2) + 4 * h2;
      if (m >= p.M) continue;
      if constexpr (SWIGLU) {
        const int n = bn * 128 + wn * 32 + c32;
        if (n >= p.pair_offset) continue;
        if (p.out32) { epi32_swiglu(p, m, n, acc[mt][0][r], acc[mt][1][r]); continue; }
        out[(size_t)m * p.ldo + n] = glu16<AT>(p.glu, acc[mt][0][r], acc[mt][1][r]);
      } else {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const int n = bn * BN2 + wn * 64 + nt * 32 + c32;
          if (n >= p.N) continue;
          if (p.out32) { epi32_plain(p, m, n, acc[mt][nt][r]); continue; }
          const float y = (float)(AT)silu_col(p.silu_cols, n, acc[mt][nt][r]);
          if (p.epi == EPI_STORE) out[(size_t)m * p.ldo + n] = (AT)y;
          else {
            AT* hh = (AT*)p.resid;
            hh[(size_t)m * p.ldo + n] = (AT)((float)hh[(size_t)m * p.ldo + n] + y);
          }
        }
      }
    }
}
#endif  // MI_GEMM_M32_BUILD

// out[row][:] = w * cast_T(x32 * rsqrt(mean(x32^2) + eps))   (nn.RMSNorm); one wave per row
template <typename AT>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const AT* x, int ldx, const AT* w, AT* out, int ldo,
                                                           int rows, int H, float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  const AT* xr = x + (size_t)row * ldx;
  float ss = 0.f;
  for (int k = lane * 8; k < H; k += 512) {
    const u32x4 v = *(const u32x4*)(xr + k);
    const AT* e = (const AT*)&v;
#pragma unroll
    for (int j = 0; j < 8; ++j) { const float f = (float)e[j]; ss = fmaf(f, f, ss); }
  }
  ss = wave_sum(ss);
  const float rs = 1.0f / sqrtf(ss / (float)H + eps);
  for (int k = lane * 8; k < H; k += 512) {
    u32x4 v = *(const u32x4*)(xr + k);
    const u32x4 wv = *(const u32x4*)(w + k);
    AT* e = (AT*)&v;
    const AT* we = (const AT*)&wv;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const AT xn = (AT)((float)e[j] * rs);
      e[j] = (AT)((float)xn * (float)we[j]);
    }
    *(u32x4*)(out + (size_t)row * ldo + k) = v;
  }
}

// The same operator with one 256-thread workgroup per row and the row held in registers (NP 16-byte pieces per
// thread): for the few rows of a decode step (gemm_skinny.hip), where one wave per row means a handful of
// workgroups walking their rows in dependent L2 round trips (9 us at 32 x 4096; this one: one round trip).
// SUMS: in front of a matrix that is multiplied as codes, with what group_sums_kernel would read back for (its additions, the same bits;
// 700 x 4096: 5.5 us and 5.9 as two launches, 5.9 as one).
template <typename AT, int NP, bool SUMS>
__global__ __launch_bounds__(256) void rmsnorm_row_block_kernel(const AT* x, int ldx, const AT* w, AT* out, int ldo, int H,
                                                                float eps, uint16_t* xs, int kb) {
  __shared__ float gsum[SUMS ? NP * 32 : 1];
  __shared__ float part[4];
  const int row = blockIdx.x, tid = threadIdx.x;
  const AT* xr = x + (size_t)row * ldx;
  u32x4 v[NP], wv[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int k = (tid + i * 256) * 8;
    const int kc = k < H ? k : 0;
    v[i] = *(const u32x4*)(xr + kc);
    wv[i] = *(const u32x4*)(w + kc);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    if ((tid + i * 256) * 8 < H) {
      const AT* e = (const AT*)&v[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) { const float f = (float)e[j]; ss = fmaf(f, f, ss); }
    }
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  const float rs = 1.0f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)H + eps);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int k = (tid + i * 256) * 8;
    if (k < H) {
      AT* e = (AT*)&v[i];
      const AT* we = (const AT*)&wv[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const AT xn = (AT)((float)e[j] * rs);
        e[j] = (AT)((float)xn * (float)we[j]);
      }
      *(u32x4*)(out + (size_t)row * ldo + k) = v[i];
      if constexpr (SUMS) {                                      // (H is a multiple of 64: a group's eight lanes are all here)
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) s += (float)e[j];
        s = lane8_sum(s);
        if ((tid & 7) == 0) gsum[k >> 6] = s;
      }
    }
  }
  if constexpr (SUMS) {
    __syncthreads();
    store_group_sums(gsum, H / 64, xs + (size_t)row * kb, kb, 1);
  }
}

// float32 storage with the run-time logical rounding (PagedKVCache mode): out = rnd(w * rnd(x * rsqrt(mean(x^2) + eps)))
__global__ __launch_bounds__(256) void rmsnorm_row_block_f32_kernel(const float* x, int ldx, const float* w, float* out, int ldo,
                                                                    int H, float eps, int rnd) {
  __shared__ float part[4];
  const int row = blockIdx.x, tid = threadIdx.x;
  const float* xr = x + (size_t)row * ldx;
  float ss = 0.f;
  for (int k = tid * 4; k < H; k += 1024) {
    const f32x4 v = *(const f32x4*)(xr + k);
    ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  const float rs = 1.0f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)H + eps);
  for (int k = tid * 4; k < H; k += 1024) {
    const f32x4 v = *(const f32x4*)(xr + k), wv = *(const f32x4*)(w + k);
    f32x4 o;
    o.x = round_rt(round_rt(v.x * rs, rnd) * wv.x, rnd);
    o.y = round_rt(round_rt(v.y * rs, rnd) * wv.y, rnd);
    o.z = round_rt(round_rt(v.z * rs, rnd) * wv.z, rnd);
    o.w = round_rt(round_rt(v.w * rs, rnd) * wv.w, rnd);
    *(f32x4*)(out + (size_t)row * ldo + k) = o;
  }
}


// float32 activations in front of the tile GEMM (PagedKVCache mode): x (optionally RMS-normalised first, in float32) is
// split EXACTLY into three 16-bit terms, x = hi + mid + lo (hi = T(x), mid = T(x - hi), lo = T(x - hi - mid): 24
// mantissa bits), stored side by side as one row [hi | mid | lo] of 3 K elements.  The GEMM then walks W three times
// (GemmParams::kw): every product is exact in the float32 accumulator, so the result is a float32 dot product in
// another summation order -- the same arithmetic as the decode step's skinny_kernel<.., X32>.  One workgroup per row.
// terms = 2 (round 4, dense bf16 weights): [hi | lo] only, 16+ mantissa bits of x, TWO walks of W instead of three.  What
// that costs in accuracy was measured on the CPU before it was built (oracle/numerics.py X_SPLIT2): the
// float32-accumulating variants' deviation from the exact oracle does not move (mean 1.91352e-4 vs 1.91362e-4).
// rnd: the normed row with the logical rounding of layer 0 (as rmsnorm_row_block_f32_kernel); values of T are one term, exactly.
template <typename AT>
__global__ __launch_bounds__(256) void split3_rows_kernel(const float* x, int ldx, const float* norm_w, float eps, AT* out,
                                                          int K, int terms, int rnd) {
  __shared__ float part[4];
  const int row = blockIdx.x, tid = threadIdx.x;
  const float* xr = x + (size_t)row * ldx;
  float rs = 1.0f;
  if (norm_w != nullptr) {
    float ss = 0.f;
    for (int k = tid * 4; k < K; k += 1024) {
      const f32x4 v = *(const f32x4*)(xr + k);
      ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    rs = 1.0f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)K + eps);
  }
  AT* o = out + (size_t)row * terms * K;
  if ((K & 7) == 0) {                                 // (uniform) 8 elements per thread and trip: 16-byte stores of every term
    for (int k = tid * 8; k < K; k += 2048) {
      f32x4 v[2] = {*(const f32x4*)(xr + k), *(const f32x4*)(xr + k + 4)};
      if (norm_w != nullptr) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 wv = *(const f32x4*)(norm_w + k + 4 * h);
#pragma unroll
          for (int j = 0; j < 4; ++j) v[h][j] = round_rt(round_rt(v[h][j] * rs, rnd) * wv[j], rnd);
        }
      }
      AT hi[8], mid[8], lo[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float xv = v[j >> 2][j & 3];
        hi[j] = (AT)xv;
        const float r1 = xv - (float)hi[j];
        mid[j] = (AT)r1;
        lo[j] = (AT)(r1 - (float)mid[j]);
      }
      *(uint4*)(o + k) = *(const uint4*)hi;
      if (terms >= 2) *(uint4*)(o + K + k) = *(const uint4*)mid;
      if (terms == 3) *(uint4*)(o + 2 * K + k) = *(const uint4*)lo;      // (uniform)
    }
    return;
  }
  for (int k = tid * 4; k < K; k += 1024) {
    f32x4 v = *(const f32x4*)(xr + k);
    if (norm_w != nullptr) {
      const f32x4 wv = *(const f32x4*)(norm_w + k);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = round_rt(round_rt(v[j] * rs, rnd) * wv[j], rnd);
    }
    AT hi[4], mid[4], lo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      hi[j] = (AT)v[j];
      const float r1 = v[j] - (float)hi[j];
      mid[j] = (AT)r1;
      lo[j] = (AT)(r1 - (float)mid[j]);
    }
    *(uint2*)(o + k) = *(const uint2*)hi;
    if (terms >= 2) *(uint2*)(o + K + k) = *(const uint2*)mid;
    if (terms == 3) *(uint2*)(o + 2 * K + k) = *(const uint2*)lo;      // (uniform)
  }
}

template <typename AT>
int launch_rmsnorm_block(const void* x, int ldx, const void* w, void* out, int ldo, int rows, int H, float eps, hipStream_t st, uint16_t* xs = nullptr, int kb = 0) {
  const int np = (H / 8 + 255) / 256;
  const dim3 grid(rows), block(256);
#define GO(NP) do { if (xs != nullptr) hipLaunchKernelGGL((rmsnorm_row_block_kernel<AT, NP, true>), grid, block, 0, st, (const AT*)x, ldx, (const AT*)w, (AT*)out, ldo, H, eps, xs, kb); \
    else hipLaunchKernelGGL((rmsnorm_row_block_kernel<AT, NP, false>), grid, block, 0, st, (const AT*)x, ldx, (const AT*)w, (AT*)out, ldo, H, eps, xs, kb); } while (0)
  switch (np) {
    case 1: GO(1); break;
    case 2: GO(2); break;
    case 3: GO(3); break;
    case 4: GO(4); break;
    default: return fail(MI_ERR_UNSUPPORTED, "rmsnorm (one workgroup per row): hidden size above 8192");
  }
#undef GO
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace

// What gemm_codes256_kernel can do at all, rows of stride ldx
static bool codes_fits(const LinearW& W, const GemvCall& c, size_t rows, size_t ldx) {
  if (!wk_is_quant(W.wk) || W.layout != 1 || W.group != 64 || W.K % BK != 0 || W.K > 65536) return false;      // (the biases of a row tile in 64 KiB of LDS)
  if (c.glu.kind != GLU_SILU || c.silu_cols > 0) return false;                 // (no quantised model has another unit)
  const size_t lim = (size_t)1 << 32;                    // (32-bit offsets of the LDS-DMA sources)
  return rows * ldx * 2 < lim && rows * codes16_bias_cols(W.K) * 2 < lim && (size_t)W.N * (W.K / 64) * 4 < lim;
}

bool gemm_prefill_supported(const LinearW& W, const GemvCall& c, size_t rows) {
  if (c.force_v1 || W.layout != 1) return false;
  // logical rounding (layer 0 of the PagedKVCache mode): plain stores of float32 activations
  if (c.rnd != RND_NONE && (c.act != MI_F32 || c.epi != EPI_STORE || W.lora_b[0] != nullptr || W.lora_b[1] != nullptr)) return false;
  if (rows < 32) return false;
  const bool dense = (W.wk == WK_BF16 && c.act == MI_BF16) || (W.wk == WK_F16 && c.act == MI_F16);
  const bool q4 = ((W.wk == WK_Q4_BF16 && c.act == MI_BF16) || (W.wk == WK_Q4_F16 && c.act == MI_F16)) && W.group == 64 &&
                  W.K % 128 == 0;                       // through a [hi | lo] 16-bit copy (launch_dequant_q4_hilo)
  const bool q8 = ((W.wk == WK_Q8_BF16 && c.act == MI_BF16) || (W.wk == WK_Q8_F16 && c.act == MI_F16)) && W.group == 64;
  // float32 activations on a bf16 model (PagedKVCache mode): x goes through launch_split3_rows first.  int8: on the codes alone (codes_plan says
  // why), and above 128 rows: up to there (a decode batch) the streaming kernel is ahead where the time is (us, streaming / codes: 64 rows
  // 6144 x 4096 41 / 69, 4096 x 14336 68 / 178, 2048 x 2048 30 / 40; 96 rows 62 / 70, 102 / 179, 45 / 42; 1024 x 1024, 96 rows 36 / 29)
  static const bool f32_ok = getenv("MI_GEMM_NO_F32") == nullptr;
  const bool x32 = f32_ok && c.act == MI_F32 && (W.wk == WK_BF16 || (W.wk == WK_Q4_BF16 && W.group == 64 && W.K % 128 == 0) ||
                                                 (W.wk == WK_Q8_BF16 && rows > 128 && codes_fits(W, c, rows, 3 * (size_t)W.K))) &&
                   c.ldx % 4 == 0 && W.K % 4 == 0;
  if (!dense && !q4 && !q8 && !x32) return false;
  if (W.K % BK != 0 || (!x32 && c.ldx % 8 != 0)) return false;
  if (c.out32 && (c.epi == EPI_SWIGLU || W.lora_b[0] || W.lora_b[1])) return false;
  // an adapted matrix: the caller adds the LoRA term to the stored output afterwards (launch_lora_up_add)
  if ((W.lora_b[0] != nullptr || W.lora_b[1] != nullptr) && c.epi != EPI_STORE) return false;
  const int n = c.epi == EPI_SWIGLU ? c.pair_offset : W.N;
  return n % 16 == 0 && (c.epi != EPI_SWIGLU || c.pair_offset % 16 == 0);
}

// Measured as whole calls of one layer and the logits of every position, float32 caches (tile GEMM minus streaming kernel, us; Mistral-7B /
// Qwen3-14B shapes):
//   rounded q|k|v, dense  33 rows -10 / -7, 128 -37 / -27, 1024 -421 / -656 (one term, one walk of W)
//                  int4   96 rows +19 / +23, 128 -7 / -13, 192 -30 / -64 (the copy of W first)
//                  f16    96 rows +28 / +25, 192 -11 / +87, 768 +127 / +328, 1024 +27 / -81, 1536 -110, 2048 -555 (three terms against two)
//   logits, dense and f16 64 rows +40 / +351, 128 -26 / -112, 192 -6 / -163, 256 -214 / -1257; f16 +111 / +796, -40 / -231, +35 / +59, -367 / -2179:
//                         a row of 128-row tiles costs three to four launches of 32 rows; from 256 rows the 256 x 256 tile runs
//           int4          64 rows +323 / +2144, 512 -103 / +88, 768 +42 / -412, 1024 -341 / -760 (the copy: 4 bytes per weight; six walks)
// (int4: figures of the [hi | lo] copy.  These lines are left with the matrices that are too small for the codes at the call's rows; the others:
// gemm_prefill_pays_codes)
bool gemm_prefill_pays(bool codes, bool hilo, bool rounded, size_t rows) {
  if (rounded) return rows > (hilo ? 1535 : codes ? 96 : 31);
  if (codes) return rows >= 1024;
  return rows >= 256 || (rows + 31) / 32 > 3 * ((rows + 127) / 128);
}

int launch_rmsnorm_rows(const void* x, int ldx, const void* w, void* out, int ldo, int rows, int H, float eps, int act,
                        hipStream_t st, bool block_per_row, int rnd) {
  if (H % 8 != 0) return fail(MI_ERR_UNSUPPORTED, "rmsnorm_rows: hidden size must be a multiple of 8");
  if (act == MI_F32) {
    hipLaunchKernelGGL(rmsnorm_row_block_f32_kernel, dim3(rows), dim3(256), 0, st, (const float*)x, ldx, (const float*)w,
                       (float*)out, ldo, H, eps, rnd);
    MI_HIP(hipGetLastError());
    return MI_OK;
  }
  if (block_per_row && H <= 8192) {
    if (act == MI_BF16) return launch_rmsnorm_block<bf16>(x, ldx, w, out, ldo, rows, H, eps, st);
    if (act == MI_F16) return launch_rmsnorm_block<f16>(x, ldx, w, out, ldo, rows, H, eps, st);
  }
  const dim3 grid((rows + 3) / 4), block(256);
  if (act == MI_BF16)
    hipLaunchKernelGGL(rmsnorm_rows_kernel<bf16>, grid, block, 0, st, (const bf16*)x, ldx, (const bf16*)w, (bf16*)out, ldo, rows, H, eps);
  else if (act == MI_F16)
    hipLaunchKernelGGL(rmsnorm_rows_kernel<f16>, grid, block, 0, st, (const f16*)x, ldx, (const f16*)w, (f16*)out, ldo, rows, H, eps);
  else return fail(MI_ERR_UNSUPPORTED, "rmsnorm_rows: 16-bit activations only");
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// c.pro must be PRO_NONE here (the caller runs launch_rmsnorm_rows first); rows = total rows of x.
// int4 weights: `scratch` (>= dequant_hilo_bytes(N, K)) receives the [hi | lo] copy first.
size_t split3_bytes(size_t rows, int K) { return rows * 3 * (size_t)K * 2; }

int launch_split3_rows(const void* x, int ldx, const void* norm_w, float eps, void* out, int rows, int K, hipStream_t st,
                       int terms, int rnd) {
  if (K % 4 != 0 || ldx % 4 != 0) return fail(MI_ERR_UNSUPPORTED, "split3_rows: K and the row stride must be multiples of 4");
  if (terms < 1 || terms > 3) return fail(MI_ERR_INVALID, "split3_rows: one to three terms");
  hipLaunchKernelGGL(split3_rows_kernel<bf16>, dim3(rows), dim3(256), 0, st, (const float*)x, ldx, (const float*)norm_w, eps,
                     (bf16*)out, K, terms, rnd);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// K slices of a 256 x 256 tile launch over `blocks` tiles: one 128-KiB workgroup per CU, so the launch runs in rounds of n_cu workgroups.  The
// split whose last round is fullest, charging 2 % per extra slice for its partial tile and its share of the reduce (q|k|v at 1024 rows: 96
// tiles -> 5 slices = 480 workgroups, 1.9 rounds; o_proj: 64 tiles -> 4 slices = one full round); at least 8 K tiles per slice.
static int split256(long blocks, int ktiles, size_t slice_bytes, size_t cap) {
  const int ncu = gemv_cu_count();
  double best = 0.0;
  int ks256 = 1;
  for (int ks = 1; ks <= 8; ++ks) {
    if (ks > 1 && (ktiles / ks < 8 || (size_t)ks * slice_bytes > cap)) break;
    const long wgs = blocks * ks, rounds = (wgs + ncu - 1) / ncu;
    const double score = (double)wgs / (double)(rounds * ncu) * (1.0 - 0.02 * (ks - 1));
    if (score > best + 1e-9) { best = score; ks256 = ks; }
  }
  return ks256;
}

// 16-byte pieces of the output rows (and of the residual's): strides and bases of float or AT elements (split_out: 8 bytes of bf16)
static int strips_ok(const GemmParams& p) {
  const void* dst = p.epi == EPI_RESID ? p.resid : p.out;
  return p.ldo % (p.out32 ? 4 : 8) == 0 && ((uintptr_t)dst & 15) == 0;
}

static int reduce_slices(const GemmParams& p, int act, hipStream_t st) {
  const size_t total4 = (size_t)p.M * p.N / 4;
  const dim3 rg((unsigned)((total4 + 255) / 256));
  if (act == MI_F16) hipLaunchKernelGGL(splitk_epilogue_kernel<f16>, rg, dim3(256), 0, st, p);
  else hipLaunchKernelGGL(splitk_epilogue_kernel<bf16>, rg, dim3(256), 0, st, p);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

size_t gemm_prefill_scratch_bytes(const LinearW& W, const GemvCall& c, size_t rows) {
  const size_t sums = rows * codes16_bias_cols(W.K) * 2;
  if (c.codes && W.codes.codes != nullptr) return sums;          // (the copy is kept)
  return std::max(dequant_hilo_bytes(W.N, W.K), codes16_bytes(W.N, W.K) + sums);
}

// us of a launch over `blocks` tiles of `nk` K tiles in rounds of one workgroup per CU, those from `tail` on as `ks` slices.  16-bit rows: a full round 10 + 2 per K tile; one that leaves
// CUs idle has the power that they do not draw, 0.72 to 0.92 of that per K tile; what joins the slices 3 + 0.09 each (writing 256 KiB at the end of the loop, and reading them).  Prompts of
// one document through six layers, int4, us a layer that slices give, by this and measured: 48 tiles (3072 x 4096, 300 rows) 56 / 52, 72 tiles 44 / 41, 120 26 / 24, 88 32 / 32, 336 (14336 x
// 4096, 700 rows) 52 / 35, 272 (17408 x 5120, 512 rows) 96 / 88, 88 of 35 K tiles (5632 x 2048) 6 / 9; none by this: 144 tiles -10, 132 -6, 408 -8, 680 -8 (they were sliced while every
// round counted as a full one).  Float32 rows: 1.35 per K tile, as their three walks find W and x in the caches, and 256 KiB at 4.9 TB/s.
static double tail_us(long blocks, long tail, int nk, int ks, bool x3, int ncu) {
  const auto rounds = [&](long n, int tiles) {
    const long part = n % ncu;
    const double tile = x3 ? 1.35 : 2.0;
    return (double)(n / ncu) * (10.0 + tile * tiles) + (part > 0 ? 10.0 + tile * tiles * (x3 ? 1.0 : 0.72 + 0.2 * part / ncu) : 0.0);
  };
  if (tail == blocks) return rounds(blocks, nk);
  const long slices = (blocks - tail) * ks;
  return rounds(tail, nk) + rounds(slices, (nk + ks - 1) / ks) + 3.0 + slices * (x3 ? 0.262144 / 4.9 : 0.09);
}

// K slices for the tiles of a last, partly filled round (all of them where there is only that round) of a call that split256 leaves whole: the cheapest by the line above, at least
// 8 K tiles a slice.  Whole columns of tiles: all rows of a call have one order of sums.  700 rows, us: 28672 x 4096 SwiGLU (336 tiles, the last 81 in three) 277 -> 200 + 16.
// Calls that split256 splits keep its slices.  Fewer of them, or of the last tiles alone, are faster (6144 x 4096, 700 rows: three for seven 54 + 13 us against 66 + 23), but an output's
// chain of additions is as long as its slice: float32 rows 1.8e-7 from 64 bits in 2-norm for 1.2e-7, and of 16-bit results 14 % more rounded the other way.
// Float32 rows take three slices or more: with two, x's largest term, which is walked last, stays one chain and the join is a rounding more (2-norm from 64 bits against the unsplit call,
// 28672 x 4096, 64 rows 1.008, 12800 x 2048, 300 rows 1.02, 6144 x 1024, 1024 rows 1.03; three to eight slices 0.78 to 1.00 over 4 shapes and 7 row counts).
static void tail_plan(long mb, long blocks, int nk, bool x3, size_t cap, GemmParams& p) {
  const int ncu = gemv_cu_count();
  double best = tail_us(blocks, blocks, nk, 1, x3, ncu) - (x3 ? 10.0 : 5.0);       // (what the line is sure of)
  for (const long tail : {blocks / ncu * ncu / mb * mb, 0L}) {
    for (int ks = x3 ? 3 : 2; ks <= 8 && nk / ks >= 8 && (size_t)(blocks - tail) * ks * (BM2 * BN2 * 4) <= cap; ++ks) {
      if (tail == blocks) break;
      const double t = tail_us(blocks, tail, nk, ks, x3, ncu);
      if (t < best) { best = t; p.mb = (int)mb; p.tail = (int)tail; p.ksplit = ks; }
    }
  }
}

// Does gemm_codes256_kernel take this call of a quantised matrix?  It halves the products and the copy of the [hi | lo] form and costs a launch (the
// group sums), the bias columns and a 256-row tile where the other has 128.  Whole calls, us, codes and [hi | lo], bf16 rows: 4096 x 4096 x
// 129 rows 43 / 50, 28672 x 4096 SwiGLU 129 rows 196 / 317 and 700 rows 348 / 494, 4096 x 14336 x 700 144 / 221; 2048 x 5632 x 192 44 / 41, 256 44 / 50;
// 4096 x 2048 x 768 47 / 53, 1536 59 / 101; 2048 x 1024 x 2048 43 / 43, 4096 57 / 55; 6144 x 1024 SwiGLU 768 57 / 54, 1536 60 / 82.  Float32 rows
// (three walks against six): 2048 x 1024 x 768 42 / 42, 1536 55 / 62; 3072 x 1024 x 768 49 / 58.
// Int8 on float32 rows at any size: the alternative there is the streaming kernel on exact codes, and a pair of bf16 is no match for it once a group's
// mean exceeds 3 of its deviations.  2-norm from 64 bits, 1024 x 1024, 256 rows, means of 0 / 4 / 12 deviations: pair 1.8e-7 / 7.0e-7 / 1.9e-6,
// streaming 3.3e-7 / 1.3e-7 / 1.0e-7, here 0.8e-7 / 0.7e-7 / 0.7e-7 (2048 x 4096, 160 rows: 3.7e-7 / 7.7e-7 / 1.9e-6, 3.4e-7 / 1.4e-7 / 1.2e-7, 1.2e-7 / 0.8e-7 / 0.8e-7);
// us, streaming / here: 129 rows 59 / 29, 1365 rows 511 / 40.
static bool codes_plan(const LinearW& W, const GemvCall& c, size_t rows, int ldx, int terms, bool split_ok, size_t cap, GemmParams& p, long& blocks) {
  const bool sw = c.epi == EPI_SWIGLU;
  const int ncols = sw ? c.pair_offset : W.N;
  if (!codes_fits(W, c, rows, ldx)) return false;
  const bool any = c.codes || (c.act == MI_F32 && wk_bits(W.wk) == 8);
  if (!any && (double)rows * W.N * W.K * terms < (W.K >= 4096 ? 2.1e9 : 4.3e9)) return false;
  p.M = (int)rows; p.N = W.N; p.kw = W.K; p.ka = p.K = terms * W.K; p.ldx = ldx; p.G = W.K / 64;
  p.kb = codes16_bias_cols(W.K);
  blocks = (long)((rows + BM2 - 1) / BM2) * ((ncols + (sw ? 128 : BN2) - 1) / (sw ? 128 : BN2));
  p.ksplit = !sw && split_ok && W.N % 4 == 0 ? split256(blocks, (p.ka + p.kb) / BK, rows * W.N * sizeof(float), cap) : 1;
  if (split_ok && p.ksplit == 1) tail_plan((long)((rows + BM2 - 1) / BM2), blocks, (p.ka + p.kb) / BK, terms > 1, cap, p);
  return true;
}

// Float32 rows against a quantised matrix: the tile GEMM, or 32 rows per launch of the streaming kernel?  us of both, fitted to 16 shapes of int4 and int8:
// a launch of the streaming kernel 11 + 0.30 per 2^20 weights + 0.5 per 1024 columns (6144 x 4096 20, 28672 x 4096 42 int4 and 45 int8, 2048 x 6400 20, 5120 x
// 17408 54 and 57); the codes' copy 0.65, a round of workgroups 1.35 per K tile, the reduce of split256's slices.  own_copy: the call makes the copy of the codes.  The engine's calls
// leave it out of the price whether or not they have one that is kept: the kernels differ in their last bits, and a prompt's are not to depend on the memory that was free at load time.
// tail_plan's slices are not priced, so a SwiGLU stays on the streaming kernel for longer than it should.  Kernel times of both at 96 to 512 rows, 18 shapes of int4 and int8: with kept
// codes the choice is never behind where it takes the codes and 7 % behind the better side on average (streaming / codes: 12800 x 2048 SwiGLU 224 rows 170 / 69, 256 rows 194 / 69,
// taken; 28672 x 4096 SwiGLU 160 rows 226 / 210, 192 rows 271 / 214, taken; 34816 x 5120 SwiGLU 160 rows 378 / 292; 6144 x 4096 96 rows 65 / 65, 129 rows 108 / 67, both taken); with a
// copy per call 4 % (6144 x 4096 96 rows 65 / 81, 4096 x 14336 129 rows 188 / 200, both taken).
static bool gemm_prefill_pays_codes(const LinearW& W, const GemvCall& c, size_t rows, int terms, bool own_copy, size_t splitk_cap) {
  GemmParams p{};
  long blocks = 0;
  if (!codes_plan(W, c, rows, terms * W.K, terms, splitk_cap > 0, splitk_cap, p, blocks))
    return (c.rnd == RND_NONE && c.epi != EPI_STORE_F32) || gemm_prefill_pays(true, false, c.rnd != RND_NONE, rows);
  const int ks = p.mb == 0 ? p.ksplit : 1;
  const int ncu = gemv_cu_count(), tiles = ((p.ka + p.kb) / BK + ks - 1) / ks;
  const double mw = (double)W.N * W.K / (1 << 20), rounds = (double)((blocks * ks + ncu - 1) / ncu);
  const double reduce = ks > 1 ? 2e-6 * ks * rows * W.N : 0.0;
  return 12.0 + (own_copy ? 0.65 * mw : 0.0) + 1.35 * rounds * tiles + reduce < (double)((rows + 31) / 32) * (11.0 + 0.30 * mw + 0.5 * W.K / 1024);
}

bool gemm_prefill_on_codes(const LinearW& W, const GemvCall& c, size_t rows) {
  const int terms = c.act == MI_F32 && c.rnd != RND_BF16 ? 3 : 1;
  GemmParams p{};
  long blocks = 0;
  return codes_plan(W, c, rows, c.act == MI_F32 ? terms * W.K : c.ldx, terms, false, 0, p, blocks);
}

int gemm_prefill_quant_route(const LinearW& W, const GemvCall& c, size_t rows, bool own_copy) {
  if (!gemm_prefill_supported(W, c, rows)) return 0;
  const bool x32 = c.act == MI_F32;
  const int terms = x32 && c.rnd != RND_BF16 ? 3 : 1;
  const size_t cap = rows < 4096 ? (size_t)128 << 20 : 0;                       // (of the engine's workspace for slices)
  if (x32 && rows > 32 && gemm_skinny_supported(W, c, 32) && !gemm_prefill_pays_codes(W, c, rows, terms, own_copy, cap)) return 0;
  return gemm_prefill_on_codes(W, c, rows) ? 2 : 1;
}

template <typename AT, bool SWIGLU, bool LOGITS, bool X3 = false>
static int codes_launch(const GemmParams& p, dim3 grid, hipStream_t st) {
  auto k = gemm_codes256_kernel<AT, SWIGLU, LOGITS, X3>;
  static std::atomic<bool> opted_in[64];                // per device: several engines, and threads, may live in one process
  int dev = 0;
  MI_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64 || !opted_in[dev].load(std::memory_order_acquire)) {
    MI_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, CODES_LDS));
    if (dev >= 0 && dev < 64) opted_in[dev].store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(k, grid, dim3(512), CODES_LDS, st, p);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// quantised matrices on gemm_codes256_kernel; *done = false: the [hi | lo] copy and the dense tiles take the call
static int launch_gemm_codes(const LinearW& W, const GemvCall& c, size_t rows, hipStream_t st, void* scratch, void* splitk_ws, size_t splitk_cap, bool* done) {
  *done = false;
  const bool sw = c.epi == EPI_SWIGLU, x32 = c.act == MI_F32;
  const int terms = x32 ? c.ldx / W.K : 1, ncols = sw ? c.pair_offset : W.N;
  GemmParams p{};
  long blocks = 0;
  if (!codes_plan(W, c, rows, c.pro == PRO_NORM ? W.K : c.ldx, terms, splitk_ws != nullptr, splitk_cap, p, blocks)) return MI_OK;
  p.x = c.x;
  p.ws = (float*)splitk_ws;
  char* d = (char*)scratch;
  if (c.codes && W.codes.codes != nullptr) {             // (a copy that was made when the weights were loaded; gemm_prefill_scratch_bytes asks the same)
    p.w = W.codes.codes; p.wb = W.codes.bias[terms != 1]; p.sc = W.codes.scales;
  } else {
    MI_TRY(launch_codes16(W, scratch, st, terms == 1));
    p.w = d; p.wb = d + (size_t)W.N * W.K * 2; p.sc = (const float*)(d + (size_t)W.N * (W.K + p.kb) * 2);
    d += codes16_bytes(W.N, W.K);
  }
  uint16_t* xs = (uint16_t*)d;
  p.xs = xs;
  if (c.pro == PRO_NORM) {
    MI_TRY((c.act == MI_F16 ? launch_rmsnorm_block<f16> : launch_rmsnorm_block<bf16>)(c.x, c.ldx, c.norm_w, c.norm_out, W.K, (int)rows, W.K, c.eps, st, xs, p.kb));
    p.x = c.norm_out; p.ldx = W.K;
  } else if (c.act == MI_F16) hipLaunchKernelGGL(group_sums_kernel<f16>, dim3((unsigned)rows), dim3(256), p.G * sizeof(float), st, (const f16*)c.x, c.ldx, terms, W.K, xs, p.kb, terms == 1);
  else hipLaunchKernelGGL(group_sums_kernel<bf16>, dim3((unsigned)rows), dim3(256), p.G * sizeof(float), st, (const bf16*)c.x, c.ldx, terms, W.K, xs, p.kb, terms == 1);
  MI_HIP(hipGetLastError());
  p.out32 = x32 || c.out32; p.rnd = x32 ? c.rnd : RND_NONE;
  p.epi = c.epi; p.out = c.out; p.ldo = c.ldo; p.resid = c.resid; p.pair_offset = c.pair_offset; p.glu = c.glu; p.silu_cols = c.silu_cols;
  if (c.epi == EPI_STORE_F32) {
    p.epi = EPI_STORE;
    if (!x32) { p.out32 = 1; p.rnd = c.act == MI_BF16 ? RND_BF16 : RND_F16; }
  }
  p.strips = strips_ok(p);
  const dim3 grid = p.mb > 0 ? dim3((unsigned)(p.tail + (blocks - p.tail) * p.ksplit)) : dim3((unsigned)((rows + BM2 - 1) / BM2), (ncols + (sw ? 128 : BN2) - 1) / (sw ? 128 : BN2), p.ksplit);
  const bool rounded = p.rnd != RND_NONE;               // (float32 stores of values rounded to 16 bits: logits, and layer 0 of the float32-cache mode)
  if (terms > 1 && !rounded) MI_TRY((sw ? codes_launch<bf16, true, false, true> : codes_launch<bf16, false, false, true>)(p, grid, st));
  else if (c.act == MI_F16) MI_TRY((sw ? codes_launch<f16, true, false> : rounded ? codes_launch<f16, false, true> : codes_launch<f16, false, false>)(p, grid, st));
  else MI_TRY((sw ? codes_launch<bf16, true, false> : rounded ? codes_launch<bf16, false, true> : codes_launch<bf16, false, false>)(p, grid, st));
  if (p.mb == 0 && p.ksplit > 1) MI_TRY(reduce_slices(p, c.act, st));
  if (p.mb > 0) {
    const dim3 rg((unsigned)(blocks - p.tail), 8), rb(512);
#define TAIL_GO(T) do { if (sw) hipLaunchKernelGGL((tail_reduce_kernel<T, true, false>), rg, rb, 0, st, p); \
      else if (rounded) hipLaunchKernelGGL((tail_reduce_kernel<T, false, true>), rg, rb, 0, st, p); \
      else hipLaunchKernelGGL((tail_reduce_kernel<T, false, false>), rg, rb, 0, st, p); } while (0)
    if (c.act == MI_F16) TAIL_GO(f16); else TAIL_GO(bf16);
#undef TAIL_GO
    MI_HIP(hipGetLastError());
  }
  *done = true;
  return MI_OK;
}

static bool gemm_small_only() { static const bool v = getenv("MI_GEMM_TILE128") != nullptr; return v; }        // A/B: always the 128 x 128 kernel
static bool gemm_dma_on() { const char* v = getenv("MI_GEMM_DMA"); return v == nullptr || atoi(v) != 0; }      // A/B and the bit-equality test: 0 = the register-staged tile (read per call)

bool gemm_prefill_split_out(const LinearW& W, const GemvCall& c, size_t rows) {
  if (c.act != MI_F32 || c.epi != EPI_SWIGLU || c.kx > 0 || W.wk != WK_BF16 || c.pair_offset % 2 != 0 || rows < BM2) return false;
  const long blocks256 = (long)((rows + BM2 - 1) / BM2) * ((c.pair_offset + 127) / 128);
  return !gemm_small_only() && gemm_dma_on() && blocks256 >= 192 && 2 * W.K >= 2 * BK && c.ldo % 4 == 0 && ((uintptr_t)c.out & 15) == 0;
}

int launch_gemm_prefill(const LinearW& W, const GemvCall& c, size_t rows, hipStream_t st, void* scratch, void* splitk_ws,
                        size_t splitk_cap) {
  if (c.pro != PRO_NONE && !(c.norm_out != nullptr && c.codes && c.act != MI_F32 && W.K <= 8192)) return fail(MI_ERR_INVALID, "gemm_prefill: normalise the rows first");
  GemmParams p{};
  p.ksplit = 1;
  p.x = c.x; p.ldx = c.ldx; p.M = (int)rows; p.w = W.w; p.N = W.N; p.K = W.K; p.ka = W.K; p.kw = W.K;
  if (wk_is_quant(W.wk)) {
    if (scratch == nullptr) return fail(MI_ERR_INVALID, "gemm_prefill: int4 weights need a dequantisation scratch buffer");
    const bool split_ok = c.act != MI_F32 || (c.ldx % W.K == 0 && (c.ldx == 3 * W.K || (c.ldx == W.K && c.rnd == RND_BF16)));
    bool done = false;
    if (split_ok) MI_TRY(launch_gemm_codes(W, c, rows, st, scratch, splitk_ws, splitk_cap, &done));
    if (done) return MI_OK;
    if (c.codes || (c.act == MI_F32 && wk_bits(W.wk) == 8)) return fail(MI_ERR_UNSUPPORTED, "gemm_prefill: this call does not run on the codes");
    MI_TRY(launch_dequant_q4_hilo(W, scratch, st));
    p.w = scratch; p.K = 2 * W.K; p.kw = 2 * W.K;
  }
  const bool x32 = c.act == MI_F32;        // c.x is the bf16 image of launch_split3_rows, c.ldx its terms x the true K
  if (x32) {
    // c.kx > 0: W is the persistent [hi | lo] bf16 copy of an f16 matrix (2 kx columns, launch_f16_to_hilo) -- the same
    // walk as over an int4 matrix's on-the-fly [hi | lo] copy: x = [hi | mid | lo] (3 kx) against W (2 kx) over 6 kx steps
    const bool hilo = c.kx > 0 && !wk_is_quant(W.wk);
    const int kt = hilo ? c.kx : W.K;      // the true K
    if (hilo && (W.K != 2 * c.kx || W.wk != WK_BF16)) return fail(MI_ERR_INVALID, "gemm_prefill: a [hi | lo] matrix has 2 kx bf16 columns");
    const bool pair = wk_is_quant(W.wk) || hilo;     // W itself is a [hi | lo] pair: 3 x-terms against 2 W-terms meet over 6 kt steps
    const int terms = c.ldx == kt ? 1 : c.ldx == 2 * kt ? 2 : 3;
    // (one term: values that are bf16 already, i.e. the rounded call of layer 0 -- any other row of stride K is one nobody has split)
    if (c.ldx != terms * kt || (pair && terms == 2) || (terms == 1 && c.rnd != RND_BF16))
      return fail(MI_ERR_INVALID, "gemm_prefill: float32 activations must be split first (launch_split3_rows; two terms: dense bf16 weights only)");
    p.ka = terms * kt; p.K = terms * (pair ? 2 : 1) * kt; p.out32 = 1; p.rnd = c.rnd;
    if (hilo) p.kw = 2 * kt;
  }
  if (c.out32) p.out32 = 1;
  p.epi = c.epi; p.out = c.out; p.ldo = c.ldo; p.resid = c.resid; p.pair_offset = c.pair_offset;
  if (c.epi == EPI_STORE_F32) {            // logits: float32, rounded to the activation dtype first
    p.epi = EPI_STORE;
    if (!x32) { p.out32 = 1; p.rnd = c.act == MI_BF16 ? RND_BF16 : RND_F16; }
  }
  p.glu = c.glu; p.silu_cols = c.silu_cols;
  const bool sw = c.epi == EPI_SWIGLU;
  const int ncols = sw ? c.pair_offset : W.N;
  const bool small_only = gemm_small_only();
  static const bool b_in_lds = getenv("MI_GEMM_B_DIRECT") == nullptr;         // A/B: set = W fragments straight from global
  // The 256 x 256 tile only where its grid fills the chip: at 8 x 1024 rows every linear has >= 512 blocks, but one prompt
  // of 256..1024 tokens gives N/256 x (1..4) blocks -- 16..64 for N = 4096 -- and measured 25 / 25 / 30 ms for 256 / 512 /
  // 1024 tokens against 14 / 17 / 23 ms on the 128 x 128 tile (Mistral-7B bf16; tools/debug/prefill_sweep.py).
  const long blocks256 = (long)(((int)rows + BM2 - 1) / BM2) * ((ncols + (sw ? 128 : BN2) - 1) / (sw ? 128 : BN2));
  const bool dma = gemm_dma_on();
  if (c.split_out && !gemm_prefill_split_out(W, c, rows)) return fail(MI_ERR_INVALID, "gemm_prefill: this call does not store split rows");
  p.split_out = c.split_out;
  p.strips = strips_ok(p);
  // too few 256 x 256 tiles for the chip (one prompt of 256..4095 rows against N = 4096 / 6144): the LDS-DMA tile with K
  // split over up to 8 workgroups, each >= 8 K tiles (plain / residual epilogues; SwiGLU launches have enough tiles or
  // stay on the 128 x 128 kernel).  MI_GEMM_DMA_SPLITK=0 switches it off (A/B).
  int ks256 = 1;
  const char* sk_env = getenv("MI_GEMM_DMA_SPLITK");     // (read per call: the tests switch it)
  const bool splitk256 = sk_env == nullptr || atoi(sk_env) != 0;
  const bool fold = x32 && c.rnd != RND_NONE;           // (plain stores: gemm_prefill_supported)
  const bool logits = !x32 && p.rnd != RND_NONE;
  if (rows >= 256 && !small_only && !fold && dma && splitk256 && !sw && splitk_ws != nullptr && W.N % 4 == 0) {
    ks256 = split256(blocks256, p.K / BK, rows * W.N * sizeof(float), splitk_cap);
  }
  if (rows >= 256 && !small_only && !fold && (blocks256 >= 192 || ks256 > 1)) {  // both operands through LDS (256 x 256 tile)
    const int bn = sw ? 128 : BN2;
    dim3 grid2(((int)rows + BM2 - 1) / BM2, (ncols + bn - 1) / bn), block2(512);
    if (ks256 > 1) { grid2.z = ks256; p.ksplit = ks256; p.ws = (float*)splitk_ws; }
#ifdef MI_GEMM_M32_BUILD
    static const bool m32 = getenv("MI_GEMM_M32") != nullptr;               // A/B: the 32x32x16 form of the tile
#endif
    const bool use_dma = dma && p.K >= 2 * BK;
#ifdef MI_GEMM_M32_BUILD
#define GO256_M32(T, S) else if (m32) { auto k = gemm_tile256_m32_kernel<T, S>; \
        MI_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, LDS2_BYTES)); \
        hipLaunchKernelGGL(k, grid2, block2, LDS2_BYTES, st, p); }
#else
#define GO256_M32(T, S)
#endif
#define GO256(T, S, LG) do { \
      if (use_dma) { auto k = gemm_dma256_kernel<T, S, false, LG>; \
        MI_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, DMA256_LDS)); \
        hipLaunchKernelGGL(k, grid2, block2, DMA256_LDS, st, p); } \
      GO256_M32(T, S) \
      else if (b_in_lds) { auto k = gemm_tile256_kernel<T, S, false, LG>; \
        MI_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, LDS2_BYTES)); \
        hipLaunchKernelGGL(k, grid2, block2, LDS2_BYTES, st, p); } \
      else { auto k = gemm_tile256_kernel<T, S, true, LG>; \
        MI_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * A2_BYTES)); \
        hipLaunchKernelGGL(k, grid2, block2, 2 * A2_BYTES, st, p); } } while (0)
    if (c.act == MI_BF16 || x32) { if (sw) GO256(bf16, true, false); else if (logits) GO256(bf16, false, true); else GO256(bf16, false, false); }
    else { if (sw) GO256(f16, true, false); else if (logits) GO256(f16, false, true); else GO256(f16, false, false); }
#undef GO256
    MI_HIP(hipGetLastError());
    if (p.ksplit > 1) MI_TRY(reduce_slices(p, c.act, st));
    return MI_OK;
  }
  dim3 grid(((int)rows + BM - 1) / BM, (ncols + (sw ? 64 : BN) - 1) / (sw ? 64 : BN)), block(256);
  // too few (M, N) blocks for 256 CUs: split K (plain / residual epilogues; W.N % 4 == 0 for the reduce kernel)
  static const bool no_splitk = getenv("MI_GEMM_NO_SPLITK") != nullptr;
  const long blocks = (long)grid.x * grid.y;
  // ~512 workgroups of 256 threads in all (two per CU): measured against a target of 256 -- 10.5 vs 11.6 ms at 384 rows,
  // 20.0 vs 21.4 at 768, 21.4 vs 22.4 at 1024 (Mistral-7B bf16, whole prefill call)
  static const int target = getenv("MI_GEMM_SPLITK_TARGET") ? atoi(getenv("MI_GEMM_SPLITK_TARGET")) : 512;   // A/B
  if (!sw && !no_splitk && splitk_ws != nullptr && blocks < target && W.N % 4 == 0) {
    int ks = (int)std::min<long>(8, std::max<long>(1, target / blocks));
    ks = std::min(ks, (p.K / BK) / 8);                       // at least 8 K steps per slice
    while (ks > 1 && (size_t)ks * rows * W.N * sizeof(float) > splitk_cap) --ks;
    if (ks > 1) { p.ksplit = ks; p.ws = (float*)splitk_ws; grid.z = ks; }
  }
  if (fold) hipLaunchKernelGGL((gemm_tile_kernel<bf16, false, false, true>), grid, block, 0, st, p);
  else if (c.act == MI_BF16 || x32) {
    if (sw) hipLaunchKernelGGL((gemm_tile_kernel<bf16, true>), grid, block, 0, st, p);
    else if (logits) hipLaunchKernelGGL((gemm_tile_kernel<bf16, false, false, false, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((gemm_tile_kernel<bf16, false>), grid, block, 0, st, p);
  } else {
    if (sw) hipLaunchKernelGGL((gemm_tile_kernel<f16, true>), grid, block, 0, st, p);
    else if (logits) hipLaunchKernelGGL((gemm_tile_kernel<f16, false, false, false, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((gemm_tile_kernel<f16, false>), grid, block, 0, st, p);
  }
  MI_HIP(hipGetLastError());
  if (p.ksplit > 1) MI_TRY(reduce_slices(p, c.act, st));
  return MI_OK;
}

int launch_gemm_grouped(const GroupedGemm& g, hipStream_t st) {
  const bool dense = (g.W.wk == WK_BF16 && g.act == MI_BF16) || (g.W.wk == WK_F16 && g.act == MI_F16);
  const bool last = g.last.w != nullptr;
  if (!dense || g.W.layout != 1 || g.W.K % BK != 0 || g.ldx % 8 != 0 || g.ldo % 8 != 0 || g.rows % 32 != 0 || g.W.N != g.rows * g.groups ||
      (last && (g.last.wk != g.W.wk || g.last.layout != 1 || g.last.K % BK != 0 || g.last.N % 32 != 0)))
    return fail(MI_ERR_UNSUPPORTED, "gemm_grouped: shape / layout not supported");
  GemmParams p{};
  p.ksplit = 1;
  p.x = g.x; p.ldx = g.ldx; p.w = g.W.w; p.N = g.rows; p.K = p.ka = p.kw = g.W.K;
  p.epi = EPI_STORE; p.out = g.out; p.ldo = g.ldo; p.glu = g.glu;
  p.tiles = g.tiles; p.x_rows = g.x_rows; p.out_rows = g.out_rows; p.groups = g.groups;
  p.w_last = g.last.w; p.N_last = last ? g.last.N : 0; p.K_last = last ? g.last.K : 0;
  const int cols = std::max(g.rows, p.N_last) / (g.swiglu ? 2 : 1);
  if (g.tile == BM2) {
    if (g.W.K < 2 * BK || (last && g.last.K < 2 * BK)) return fail(MI_ERR_UNSUPPORTED, "gemm_grouped: the 256 x 256 tile needs two K tiles");
    const dim3 grid(g.max_tiles, (cols + (g.swiglu ? 128 : BN2) - 1) / (g.swiglu ? 128 : BN2)), block(512);
    auto go = [&](auto k) -> int {
      MI_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, DMA256_LDS));
      hipLaunchKernelGGL(k, grid, block, DMA256_LDS, st, p);
      MI_HIP(hipGetLastError());
      return MI_OK;
    };
    if (g.act == MI_BF16) return g.swiglu ? go(gemm_dma256_kernel<bf16, true, true>) : go(gemm_dma256_kernel<bf16, false, true>);
    return g.swiglu ? go(gemm_dma256_kernel<f16, true, true>) : go(gemm_dma256_kernel<f16, false, true>);
  }
  if (g.tile != BM) return fail(MI_ERR_INVALID, "gemm_grouped: tiles of 128 or 256 places");
  const dim3 grid(g.max_tiles, (cols + (g.swiglu ? 64 : BN) - 1) / (g.swiglu ? 64 : BN)), block(256);
  if (g.act == MI_BF16) {
    if (g.swiglu) hipLaunchKernelGGL((gemm_tile_kernel<bf16, true, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((gemm_tile_kernel<bf16, false, true>), grid, block, 0, st, p);
  } else {
    if (g.swiglu) hipLaunchKernelGGL((gemm_tile_kernel<f16, true, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((gemm_tile_kernel<f16, false, true>), grid, block, 0, st, p);
  }
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
