// gemm_q4.hip -- nn.QuantizedLinear (MLX-affine int4, group 64: mlx_parallm/utils.py:679-690; call sites llama.py:64-67,93,143,
// 160-165,250-252; qwen3.py:37-40,63,115) for 17..128 rows of 16-bit activations: y[M][N] = x[M][K] . W_hat[N][K]^T, residual / SwiGLU /
// float32-logits / LoRA epilogues.
//
// What bounds this size is the arithmetic around the weights: per 16 columns, 64 k and 64 rows 8 matrix instructions (128 cycles), 16 unpacking
// and 16 scaling instructions (128 cycles), and they overlap only in part.  So:
//   * a workgroup is 8 waves = 2 column halves x 4 K lanes, one workgroup per CU: every SIMD has two waves with the same work.  A wave carries
//     TN = 4 or 5 column tiles (SwiGLU: the same gate or up tiles), so that a fragment of x that it reads from LDS feeds as many tiles, and every 4th
//     block of 128 k.  Nothing but x is shared, between the two halves.
//   * x and weights come by LDS-DMA: no staging registers, no loads in inline asm that the compiler could mistake for done.  x is prepared once
//     per launch (q4_prep_kernel): fragment order, nibble order, RMSNorm, sums per group.  A wave's weights of block i + 1 arrive while block i
//     is multiplied, the x of a step (64 k) one step ahead.
//   * The halves take turns: while one reads its step's x and codes into registers and issues its copies, the other multiplies (the second half
//     enters through one extra barrier).  In step, all eight waves read and then all multiply: 40960 x 5120, 64 rows, 52 us against 45.
//   * y += s sum (16 + q) x needs -16 sum x: that is the matrix instruction's C operand (prepared as float32, read once per step for 5 tiles).
//     sum_g b_g sum x is a product of its own, 32 groups (16 blocks) per instruction: the group's biases as they are loaded against the sums in
//     three bf16 terms (exact), 12 per tile and 16 blocks of 256 -- where v_mfma_f32_16x16x4_f32 on two groups a time took half of the
//     matrix core's time again.
//   * the K lanes meet in LDS, every wave adds and finishes its share of the output tiles.  Narrow linears split K over workgroups on top
//     (partial tiles, the last one to arrive adds them in slice order).
#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gemv_phase.h"

namespace mi {

int gemv_cu_count();

namespace {

using namespace gemv;

// Five column tiles a wave: the most whose accumulators and biases fit 256 registers, and for wide matrices the fewest rounds of workgroups (34816 x 5120 SwiGLU 218
// workgroups, four tiles 272: two rounds).  Where four take no more rounds a workgroup has less to do (28672 x 4096: 224 of 256 CUs instead of 180): q4_tiles.
constexpr int TW = 2, KW = 4, NW = TW * KW, RT = 2;       // (RT: column tiles of a workgroup of q4_rows_kernel)
constexpr int w_slot(int tn) { return tn * (1024 + 128); }       // codes of the tiles, then their scales | biases (64 + 64 bytes)
constexpr int Q4_LDS = 160 * 1024;

struct Q4Params {
  const void* xq; const float* sx; const float* sxo;            // prepared activations: [slab][K/64][2][MT] KiB, sums [slab][K/64][16 MT], -16 x sums [slab][K/64][64]
  int M, G;
  const void* w;
  int epi; void* out; int ldo; void* resid; int pair_tiles;
  int out_frag;                                                 // SwiGLU: out in q4_frag_elem's order
  int ntu, ntiles;                                              // column tiles of a half of the matrix (SwiGLU: gate tiles), of all of it
  int wgs;                                                      // (q4_rows_kernel: without those that only load)
  int nblk, ksplit, nslab, ngroups, nunits;                              // K / 128; units = tile groups x ksplit
  float* ws; unsigned* ctr;
  const float* lora_t; int lora_t_ld;
  const float* lora_b0; const float* lora_b1;
  int lora_row0_0, lora_n_0, lora_rank_0; float lora_scale_0;
  int lora_row0_1, lora_n_1, lora_rank_1; float lora_scale_1;
};

__device__ __forceinline__ size_t swiglu_at(const Q4Params& p, int row, int n) {       // (uniform)
  return p.out_frag > 0 ? q4_frag_elem(row, n, p.out_frag, p.ntu / 4) : (size_t)row * p.ldo + n;
}

// One workgroup per row (rows padded to whole slabs with zeros) and gridDim.y pieces of K (one with a norm: it needs the whole row).  The 8 k of dword d
// of a group (k = 64 grp + 8 d ..) are what lane group d >> 1 multiplies in step d & 1, in unpack_q4's order.
// NP > 0: a norm in front and K <= 2048 NP: the row and the norm's weights in registers, asked for at once (in loops, x once for the sum of squares and once more,
// a thread had six dependent trips to L2: 64 x 5120 5.85 us, now 5.1).
template <typename AT, int NP>
__global__ __launch_bounds__(256) void q4_prep_kernel(const AT* x, int ldx, int M, int MT, int K, const AT* norm_w, float eps, AT* xq, float* sx, float* sxo) {
  __shared__ float part[4];
  // (neighbouring rows on one XCD under round-robin placement: their pieces share the lines of a fragment.  The grid is a multiple of 16.  64 x 5120 without a norm 5.1 us in order, 4.8)
  const int row = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3), tid = threadIdx.x, MB = 16 * MT, slab = row / MB, r = row - slab * MB, G = K / 64;
  const bool live = row < M;
  const AT* xr = x + (size_t)(live ? row : 0) * ldx;
  const auto squares = [](u32x4 v, float ss) {
    const AT* e = (const AT*)&v;
#pragma unroll
    for (int j = 0; j < 8; ++j) { const float f = (float)e[j]; ss = fmaf(f, f, ss); }
    return ss;
  };
  const auto row_scale = [&](float ss) {
    ss = wave_sum(ss);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    return 1.0f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)K + eps);
  };
  const auto normed = [](u32x4 v, u32x4 wv, float rs) {
    AT* e = (AT*)&v;
    const AT* we = (const AT*)&wv;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const AT xn = (AT)((float)e[j] * rs);
      e[j] = (AT)((float)xn * (float)we[j]);
    }
    return v;
  };
  const auto put = [&](int k, u32x4 v) {
    const AT* e = (const AT*)&v;
    AT t2[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) { t2[2 * q] = e[q]; t2[2 * q + 1] = e[q + 4]; }
    const int grp = k >> 6, d = (k >> 3) & 7;
    const size_t frag = (((size_t)slab * G + grp) * 2 + (d & 1)) * MT + (r >> 4);
    *(u32x4*)((char*)xq + (frag * 64 + (d >> 1) * 16 + (r & 15)) * 16) = *(const u32x4*)t2;
    if (sx == nullptr) return;                                   // (uniform: q4_rows_kernel makes its own sums)
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) sum += (float)e[j];
    sum = lane8_sum(sum);
    if ((tid & 7) == 0) {
      sx[((size_t)slab * G + grp) * MB + r] = sum;
      sxo[((size_t)slab * G + grp) * 64 + r] = -Magic<AT>::offs * sum;
    }
  };
  const u32x4 none = {0u, 0u, 0u, 0u};
  if constexpr (NP > 0) {
    u32x4 v[NP], wv[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int k = (tid + i * 256) * 8, kc = k < K ? k : 0;
      v[i] = *(const u32x4*)(xr + kc);
      wv[i] = *(const u32x4*)(norm_w + kc);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if ((tid + i * 256) * 8 < K) ss = squares(v[i], ss);
    const float rs = row_scale(ss);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int k = (tid + i * 256) * 8;
      if (k < K) put(k, live ? normed(v[i], wv[i], rs) : none);
    }
  } else {
    float rs = 1.0f;
    if (norm_w != nullptr) {
      float ss = 0.f;
      if (live)
        for (int k = tid * 8; k < K; k += 2048) ss = squares(*(const u32x4*)(xr + k), ss);
      rs = row_scale(ss);
    }
    for (int k = (blockIdx.y * 256 + tid) * 8; k < K; k += 2048 * gridDim.y) {
      u32x4 v = none;
      if (live) {
        v = *(const u32x4*)(xr + k);
        if (norm_w != nullptr) v = normed(v, *(const u32x4*)(norm_w + k), rs);
      }
      put(k, v);
    }
  }
}

template <typename AT>
void q4_prep_launch(const GemvCall& c, dim3 grid, int rows, int mt, int K, const void* nw, void* xq, float* sx, float* sxo, hipStream_t st) {
#define PREP(NP) hipLaunchKernelGGL((q4_prep_kernel<AT, NP>), grid, dim3(256), 0, st, (const AT*)c.x, c.ldx, rows, mt, K, (const AT*)nw, c.eps, (AT*)xq, sx, sxo)
  switch (nw != nullptr ? (K + 2047) / 2048 : 0) {
    case 1: PREP(1); break;
    case 2: PREP(2); break;
    case 3: PREP(3); break;
    case 4: PREP(4); break;
    default: PREP(0);
  }
#undef PREP
}

__device__ __forceinline__ void dma16(const void* base, uint32_t off, unsigned lds) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(off), "s"(base), "s"(lds) : "memory");
}
typedef __attribute__((address_space(3))) unsigned char lds_byte;
template <typename T> using lds_ptr = __attribute__((address_space(3))) const T*;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <typename AT, int MT, bool SWIGLU, int TN>
__global__ __launch_bounds__(512, 2) void q4_kernel(const Q4Params p) {
  constexpr int W_SLOT = w_slot(TN);
  constexpr int MB = 16 * MT, X_HALF = MT * 1024, X_BUF = KW * 2 * X_HALF, X_DMAS = MT, W_DMAS = TN + 1;
  constexpr bool OFFS = std::is_same<AT, bf16>::value;          // (f16: the codes are unpacked without an offset)
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kw = wave & 3, tw = wave >> 2;
  // blocks [8 nslab j, ..): the slabs of 8 units, 8 block ids apart (one XCD under round-robin placement: the later reader finds the weights in that L2)
  int bid = blockIdx.x, slab = 0;
  if (p.nslab > 1) {
    const int per = 8 * p.nslab, blk = bid / per, rem = bid - blk * per;
    slab = rem >> 3;
    bid = blk * 8 + (rem & 7);
  }
  if (bid >= p.nunits) return;                                  // (grid padding: the whole workgroup leaves before any barrier)
  const int grp = __builtin_amdgcn_readfirstlane(bid / p.ksplit), s = __builtin_amdgcn_readfirstlane(bid - grp * p.ksplit);
  slab = __builtin_amdgcn_readfirstlane(slab);
  const int row0 = slab * MB, nblk = p.nblk;
  const int b0 = __builtin_amdgcn_readfirstlane((int)((unsigned)(s * nblk) / (unsigned)p.ksplit));
  const int b1 = __builtin_amdgcn_readfirstlane((int)((unsigned)((s + 1) * nblk) / (unsigned)p.ksplit));
  const int nit = (b1 - b0 + KW - 1) / KW, mine = max(0, (b1 - b0 - kw + KW - 1) / KW);      // steps in pairs; this lane's blocks

  // column tile a of half h (SwiGLU: of the gate or the up matrix); past the last one: the last one, never stored
  auto tile_of = [&](int h, int a) {
    if constexpr (SWIGLU) return min(grp * TN + a, p.ntu - 1) + h * p.pair_tiles;
    else return min((grp * TW + h) * TN + a, p.ntiles - 1);
  };
  const unsigned lds0 = (unsigned)(size_t)(lds_byte*)smem;
  const unsigned sum_lds = lds0 + 2 * X_BUF + kw * 1024, w_lds = lds0 + 2 * X_BUF + KW * 1024 + wave * 2 * W_SLOT;
  static_assert(2 * 4 * 2 * 4096 + KW * 1024 + NW * 2 * W_SLOT <= Q4_LDS, "x, sums, weights");

  // ---- DMA: steps are 64 k (step st = block st / 2 of this lane, group st % 2), clamped to the lane's last block (spare copies, never multiplied)
  const uint32_t lane16 = lane * 16;
  const char* gx = (const char*)p.xq + ((size_t)slab * p.G * 2 + tw) * X_HALF;
  const char* gs = (const char*)p.sxo + (size_t)slab * p.G * 256;
  const char* gw = (const char*)p.w;
  uint32_t wtile[TN];
#pragma unroll
  for (int a = 0; a < TN; ++a) wtile[a] = (uint32_t)tile_of(tw, a) * (uint32_t)nblk * 1152u;      // (uniform)
  const uint32_t sboff = (uint32_t)tile_of(tw, min(lane >> 3, TN - 1)) * (uint32_t)nblk * 1152u + 1024 + (lane & 7) * 16;     // lane: 16 bytes of tile lane / 8
  asm volatile("" : "+s"(gx), "+s"(gs), "+s"(gw));              // (in registers before the loop: a pending load of an argument makes the compiler wait for LDS reads with it)
  auto block_of = [&](int i) { return min(b0 + kw + KW * min(i, max(mine - 1, 0)), nblk - 1); };
  auto issue_x = [&](int st) {
    const uint32_t grp64 = 2 * block_of(st >> 1) + (st & 1);
    const char* src = gx + (size_t)grp64 * (2 * X_HALF);
    const unsigned dst = lds0 + (st & 1) * X_BUF + (kw * 2 + tw) * X_HALF;
#pragma unroll
    for (int m = 0; m < MT; ++m) dma16(src + m * 1024, lane16, dst + m * 1024);
  };
  auto issue_w = [&](int i) {
    const char* src = gw + (size_t)(uint32_t)block_of(i) * 1152;
    const unsigned dst = w_lds + (i & 1) * W_SLOT;
#pragma unroll
    for (int a = 0; a < TN; ++a) dma16(src + wtile[a], lane16, dst + a * 1024);
    if (lane < TN * 8) dma16(src, sboff, dst + TN * 1024);
    if (tw == 0 && lane < 32) dma16(gs + (size_t)(uint32_t)block_of(i) * 512, lane16, sum_lds + (i & 1) * 512);       // (for both halves)
  };

  f32x4 acc[TN][MT];
  uint32_t bb[TN][4];                                            // the biases of 16 blocks: lane group g holds blocks 4 g .. 4 g + 3, two groups each
#pragma unroll
  for (int a = 0; a < TN; ++a) {
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[a][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) bb[a][j] = 0u;
  }

  const unsigned code_off = ((g >> 1) * 16 + c16) * 16 + (g & 1) * 8;
  // component c (0..7) of the fragments of two packed dwords: unpack_q4 a register at a time
  uint32_t mask = 0x00780078u, magic = 0x41804180u;
  asm("" : "+v"(mask), "+v"(magic));
  auto unpack = [&](u32x2 v, int c) -> uint32_t {
    const uint32_t q = c < 4 ? v.x : v.y;
    if constexpr (std::is_same<AT, bf16>::value) return ((c & 3) == 0 ? q << 3 : (c & 3) == 1 ? q >> 1 : (c & 3) == 2 ? q >> 5 : q >> 9) & mask | magic;
    else return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, ((q >> (4 * (c & 3))) & 0x000F000Fu) | 0x64006400u) - f16x2{(_Float16)1024.f, (_Float16)1024.f});
  };
  // The sums of the last tile wait for their FMAs until the next step's first products are under way
  f32x4 d[2][MT];
  float scale[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) d[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto fold2 = [&](int a, int pa, int q) {                       // quarter-tiles: two of the FMAs of tile a
    const int m = q >> 1, r = (q & 1) * 2;
    acc[a][m][r] = fmaf(scale[pa], d[pa][m][r], acc[a][m][r]);
    acc[a][m][r + 1] = fmaf(scale[pa], d[pa][m][r + 1], acc[a][m][r + 1]);
    asm volatile("" : "+v"(acc[a][m]));                          // (here, not sunk behind the barriers)
  };
  auto step = [&](int st, int i, auto sgt, bool work) __attribute__((always_inline)) {
    constexpr int SG = decltype(sgt)::value;
    u32x4 xa[2][MT];
    f32x4 c0[MT];
    u32x2 cd[TN];
    uint32_t sd[TN];
    const unsigned xb = lds0 + SG * X_BUF + kw * 2 * X_HALF + lane16, wb = w_lds + (i & 1) * W_SLOT;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) xa[t][m] = *(lds_ptr<u32x4>)(size_t)(xb + t * X_HALF + m * 1024);
#pragma unroll
    for (int m = 0; m < MT; ++m) c0[m] = OFFS ? *(lds_ptr<f32x4>)(size_t)(sum_lds + (i & 1) * 512 + SG * 256 + (m * 16 + g * 4) * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < TN; ++a) {
      cd[a] = *(lds_ptr<u32x2>)(size_t)(wb + a * 1024 + SG * 512 + code_off);
      sd[a] = *(lds_ptr<uint32_t>)(size_t)(wb + TN * 1024 + a * 128 + c16 * 4);
    }
    if constexpr (SG == 0) {
      const bool here = work && g == ((i >> 2) & 3);
#pragma unroll
      for (int a = 0; a < TN; ++a) {
        const uint32_t bd = *(lds_ptr<uint32_t>)(size_t)(wb + TN * 1024 + a * 128 + 64 + c16 * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) bb[a][j] = here && (i & 3) == j ? bd : bb[a][j];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (tw == 0) {
      issue_x(st + 1);
      if constexpr (SG == 0) issue_w(i + 1);
      __builtin_amdgcn_s_waitcnt(0xC07F);                        // lgkmcnt(0)
    } else {
      __builtin_amdgcn_s_waitcnt(0xC07F);
      issue_x(st + 2);
      if constexpr (SG == 0) issue_w(i + 1);
      asm volatile("s_waitcnt vmcnt(%0)" :: "i"(X_DMAS + W_DMAS) : "memory");      // x of step st + 1
    }
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    if (work) {
      uint32_t w[2][8];
#pragma unroll
      for (int c = 0; c < 8; ++c) w[0][c] = unpack(cd[0], c);
      __builtin_amdgcn_sched_barrier(0);
      // behind every matrix instruction (16 cycles of the matrix core) two FMAs of the tile before and a share of the next tile's unpacking
#pragma unroll
      for (int a = 0; a < TN; ++a) {
        const int pa = (SG * TN + a) & 1;
        const u32x4 w0 = {w[a & 1][0], w[a & 1][1], w[a & 1][2], w[a & 1][3]}, w1 = {w[a & 1][4], w[a & 1][5], w[a & 1][6], w[a & 1][7]};
        if constexpr (std::is_same<AT, bf16>::value) scale[pa] = __uint_as_float(SG ? sd[a] & 0xffff0000u : sd[a] << 16);
        else scale[pa] = (float)__builtin_bit_cast(f16, (unsigned short)(sd[a] >> (16 * SG)));
#pragma unroll
        for (int k = 0; k < 2 * MT; ++k) {
          const int m = k % MT;
          d[pa][m] = k < MT ? mfma16<AT>(xa[0][m], w0, c0[m]) : mfma16<AT>(xa[1][m], w1, d[pa][m]);
          fold2(a == 0 ? TN - 1 : a - 1, pa ^ 1, k);
          if (a + 1 < TN) {
#pragma unroll
            for (int c = k * 8 / (2 * MT); c < (k + 1) * 8 / (2 * MT); ++c) w[(a + 1) & 1][c] = unpack(cd[a + 1], c);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    if (tw == 0) asm volatile("s_waitcnt vmcnt(%0)" :: "i"(SG == 0 ? W_DMAS + 1 : 0) : "memory");       // x of step st + 1, the next block's weights
    else if constexpr (SG == 1) asm volatile("s_waitcnt vmcnt(%0)" :: "i"(X_DMAS) : "memory");      // the next block's weights
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  issue_x(0); issue_w(0);
  if (tw == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else { issue_x(1); asm volatile("s_waitcnt vmcnt(%0)" :: "i"(X_DMAS) : "memory"); }
  asm volatile("s_barrier" ::: "memory");
  if (tw == 1) asm volatile("s_barrier" ::: "memory");
  for (int i0 = 0; i0 < nit; i0 += 16) {
    const int i1 = min(nit, i0 + 16);
    for (int i = i0; i < i1; ++i) {
      step(2 * i, i, std::integral_constant<int, 0>{}, i < mine);
      step(2 * i + 1, i, std::integral_constant<int, 1>{}, i < mine);
    }
    // (the last tile's sums of these blocks: the lane's last step was a second one)
#pragma unroll
    for (int k = 0; k < 2 * MT; ++k) fold2(TN - 1, (2 * TN - 1) & 1, k);
#pragma unroll
    for (int m = 0; m < MT; ++m) d[(2 * TN - 1) & 1][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    // sum_g b_g sum x over these 16 blocks: A = the sums of lane group g's 8 groups (row c16) in three bf16 terms, B = their biases
    float sums[MT][8];                                           // (all loads in one round trip: none under a condition)
    const float* sx = p.sx + (size_t)slab * p.G * MB + c16;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t at = (uint32_t)(2 * min(b0 + kw + KW * (i0 + 4 * g + (j >> 1)), nblk - 1) + (j & 1)) * MB;
#pragma unroll
      for (int m = 0; m < MT; ++m) sums[m][j] = sx[at + m * 16];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(sums[m][j]));
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      bf16 part[3][8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int i = i0 + 4 * g + (j >> 1);
        const float v = i < mine && i < i1 ? sums[m][j] : 0.f;
        const float hi = (float)(bf16)v, r = isinf(v) ? 0.f : v - hi, mid = (float)(bf16)r;
        part[0][j] = (bf16)hi; part[1][j] = (bf16)mid; part[2][j] = (bf16)(r - mid);
      }
      const u32x4 a0 = *(const u32x4*)part[0], a1 = *(const u32x4*)part[1], a2 = *(const u32x4*)part[2];
#pragma unroll
      for (int a = 0; a < TN; ++a) {
        if constexpr (std::is_same<AT, bf16>::value) {
          const u32x4 b = {bb[a][0], bb[a][1], bb[a][2], bb[a][3]};
          acc[a][m] = mfma16<bf16>(a2, b, acc[a][m]);
          acc[a][m] = mfma16<bf16>(a1, b, acc[a][m]);
          acc[a][m] = mfma16<bf16>(a0, b, acc[a][m]);
        } else {                                                 // an f16 bias is two terms of bf16
          bf16 bh[8], bl[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float v = (float)__builtin_bit_cast(f16, (unsigned short)(bb[a][j >> 1] >> (16 * (j & 1)))), hi = (float)(bf16)v;
            bh[j] = (bf16)hi;
            bl[j] = (bf16)(isinf(v) ? 0.f : v - hi);
          }
          const u32x4 h = *(const u32x4*)bh, l = *(const u32x4*)bl;
          acc[a][m] = mfma16<bf16>(a1, l, acc[a][m]);
          acc[a][m] = mfma16<bf16>(a0, l, acc[a][m]);
          acc[a][m] = mfma16<bf16>(a2, h, acc[a][m]);
          acc[a][m] = mfma16<bf16>(a1, h, acc[a][m]);
          acc[a][m] = mfma16<bf16>(a0, h, acc[a][m]);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int j = 0; j < 4; ++j) bb[a][j] = 0u;
  }
  if (tw == 0) asm volatile("s_barrier" ::: "memory");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // the spare copies have landed: the LDS is free
  __syncthreads();

  // ---- the K lanes meet: every wave leaves its sums, then takes whole output tiles (SwiGLU: pairs) in turn
  f32x4* red = (f32x4*)smem;
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[((wave * TN + a) * MT + m) * 64 + lane] = acc[a][m];
  __syncthreads();
  auto lanes_sum = [&](int h, int a, int m) {
    f32x4 v = red[((h * KW * TN + a) * MT + m) * 64 + lane];
#pragma unroll
    for (int k = 1; k < KW; ++k) v += red[(((h * KW + k) * TN + a) * MT + m) * 64 + lane];
    return v;
  };
  constexpr int HALVES = SWIGLU ? 1 : TW, UNITS = HALVES * TN * MT, PER = (UNITS + NW - 1) / NW, NV = SWIGLU ? 2 : 1;
  const int ntot = p.ntiles;
  if (p.ksplit > 1) {                                            // write-through partial tiles; the last slice to arrive adds them
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int u = wave + NW * k;
      if (u >= UNITS) break;
      const int h = u / (TN * MT), a = (u / MT) % TN, m = u % MT;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const f32x4 y = lanes_sum(SWIGLU ? v : h, a, m);
        unsigned long long* wp = (unsigned long long*)(p.ws + ((((size_t)(slab * p.ksplit + s) * (p.ngroups * TW * TN) + (grp * TW + (SWIGLU ? v : h)) * TN + a) * MT + m) * 64 + lane) * 4);
        __hip_atomic_store(wp, ((unsigned long long)__float_as_uint(y.y) << 32) | __float_as_uint(y.x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(wp + 1, ((unsigned long long)__float_as_uint(y.w) << 32) | __float_as_uint(y.z), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                                             // (also: `red` has been read)
    int* last_sh = (int*)smem;
    if (tid == 0) {
      unsigned* cp = &p.ctr[grp * p.nslab + slab];
      const unsigned old = __hip_atomic_fetch_add(cp, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = old == (unsigned)(p.ksplit - 1);
      if (last) __hip_atomic_store(cp, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last_sh = last;
    }
    __syncthreads();
    if (!*last_sh) return;
  }
  f32x4 tot[PER][NV];                                            // this wave's tiles
#pragma unroll
  for (int k = 0; k < PER; ++k)
#pragma unroll
    for (int v = 0; v < NV; ++v) tot[k][v] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (p.ksplit <= 1) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int u = min(wave + NW * k, UNITS - 1), h = u / (TN * MT), a = (u / MT) % TN, m = u % MT;
#pragma unroll
      for (int v = 0; v < NV; ++v) tot[k][v] = lanes_sum(SWIGLU ? v : h, a, m);
    }
  } else {
    for (int s0 = 0; s0 < p.ksplit; s0 += 2) {                   // (two slices of all of them per round trip)
      u32x4 pv[2][PER][NV];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < PER; ++k) {
          const int u = min(wave + NW * k, UNITS - 1), h = u / (TN * MT), a = (u / MT) % TN, m = u % MT;
#pragma unroll
          for (int v = 0; v < NV; ++v)
            pv[j][k][v] = load16_agent(p.ws + ((((size_t)(slab * p.ksplit + min(s0 + j, p.ksplit - 1)) * (p.ngroups * TW * TN) + (grp * TW + (SWIGLU ? v : h)) * TN + a) * MT + m) * 64 + lane) * 4);
        }
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (s0 + j < p.ksplit) {
#pragma unroll
          for (int k = 0; k < PER; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v)
#pragma unroll
              for (int r = 0; r < 4; ++r) tot[k][v][r] += __uint_as_float(pv[j][k][v][r]);
        }
    }
  }

  // ---- epilogue: lane (c16, g) holds y[row0 + 16 m + 4 g + r][16 tile + c16]
  AT* out = (AT*)p.out;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int u = wave + NW * k;
    if (u >= UNITS) break;
    const int h = u / (TN * MT), a = (u / MT) % TN, m = u % MT;
    if ((SWIGLU ? grp * TN + a >= p.ntu : (grp * TW + h) * TN + a >= ntot)) continue;
    const int n = tile_of(h, a) * 16 + c16;
    if constexpr (SWIGLU) {
      const f32x4 gt = tot[k][0], up = tot[k][NV - 1];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + m * 16 + g * 4 + r;
        if (row < p.M) out[swiglu_at(p, row, n)] = silu16<AT>(gt[r], up[r]);
      }
    } else {
      const f32x4 v = tot[k][0];
      float hres[4];
      if (p.epi == EPI_RESID) {
#pragma unroll
        for (int r = 0; r < 4; ++r) hres[r] = (float)((const AT*)p.resid)[(size_t)min(row0 + m * 16 + g * 4 + r, p.M - 1) * p.ldo + n];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + m * 16 + g * 4 + r;
        if (row >= p.M) continue;
        float y = (float)(AT)v[r];
        if (p.lora_t != nullptr) {
#pragma unroll
          for (int sl = 0; sl < 2; ++sl) {
            const int r0 = sl ? p.lora_row0_1 : p.lora_row0_0, ln = sl ? p.lora_n_1 : p.lora_n_0, rk = sl ? p.lora_rank_1 : p.lora_rank_0;
            const float* lb = sl ? p.lora_b1 : p.lora_b0;
            if (lb != nullptr && n >= r0 && n < r0 + ln) {
              const float z = (sl ? p.lora_scale_1 : p.lora_scale_0) * lora_dot(p.lora_t + (size_t)row * p.lora_t_ld + sl * (p.lora_t_ld / 2), lb + (n - r0), ln, rk);
              y = (float)(AT)(y + (float)(AT)z);
            }
          }
        }
        if (p.epi == EPI_STORE) out[(size_t)row * p.ldo + n] = (AT)y;
        else if (p.epi == EPI_STORE_F32) ((float*)p.out)[(size_t)row * p.ldo + n] = y;
        else ((AT*)p.resid)[(size_t)row * p.ldo + n] = (AT)(hres[r] + y);
      }
    }
  }
}

// Narrow matrices (q|k|v, o, down: 17..128 rows).  The kernel above cuts their K over workgroups, and the partial tiles' way through memory costs more than
// the products (7168 x 5120, 64 rows: 9 us behind a loop of 11).  Here a workgroup owns two column tiles (SwiGLU: a gate tile and its up tile) and all of K:
// wave w takes the blocks of 128 k w, w + 8, ..  Every fragment of x goes to one wave of the workgroup, so it comes from L2 straight into registers (whole KiB
// of prepared fragments: 70 bytes a clock and CU; the 16 rows of a fragment read from x itself: 17), and the loop has neither LDS nor barriers.  A block's
// loads go out as the last one's registers come free.  Results return in order, so x brings the codes asked for before it with it: a workgroup keeps no more
// than a block a wave in flight, and CUs without a unit read the codes ahead into the XCD's L2 (5120 x 5120 in a cold pass 16.5 us without, 14.2).
// sum x comes from the matrix core (a fragment of -16, or of ones where codes have no offset): it is the C operand of the codes' product and the biases' factor.
template <typename AT, int MT, bool SWIGLU>
__global__ __launch_bounds__(512, 2) void q4_rows_kernel(const Q4Params p) {
  constexpr int T = RT, X_HALF = MT * 1024;
  constexpr bool OFFS = std::is_same<AT, bf16>::value;          // (f16: the codes are unpacked without an offset)
  __shared__ f32x4 red[NW * T * MT * 64];
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bid = blockIdx.x, slab = 0;
  if (bid >= p.wgs) {                                            // CUs that the units leave idle bring the codes into their XCD's L2, in the order of their use
    const int xcd = bid & 7, first = p.wgs + ((xcd - p.wgs) & 7), helpers = ((int)gridDim.x - first + 7) >> 3, units = (p.nunits - xcd + 7) >> 3;
    const int rounds = (p.nblk + NW - 1) / NW, end = p.nblk * 1152;
    u32x4 any = {0u, 0u, 0u, 0u};
    for (int i = (bid - first) >> 3; i < rounds * units; i += helpers) {
      const int rd = i / units, u = (i - rd * units) * 8 + xcd;
#pragma unroll
      for (int a = 0; a < T; ++a) {
        const char* w = (const char*)p.w + (size_t)(SWIGLU ? u + a * p.pair_tiles : min(u * T + a, p.ntiles - 1)) * end;
#pragma unroll
        for (int j = 0; j < 2; ++j) any |= *(const u32x4*)(w + min(rd * NW * 1152 + min(j * 8192 + tid * 16, NW * 1152 - 16), end - 16));
      }
    }
    asm volatile("" :: "v"(any));
    return;
  }
  if (p.nslab > 1) {                                            // (slabs of a unit 8 block ids apart, as above)
    const int per = 8 * p.nslab, blk = bid / per, rem = bid - blk * per;
    slab = rem >> 3;
    bid = blk * 8 + (rem & 7);
  }
  if (bid >= p.nunits) return;
  const int unit = __builtin_amdgcn_readfirstlane(bid), row0 = __builtin_amdgcn_readfirstlane(slab) * 16 * MT;
  const int mine = (p.nblk - wave + NW - 1) / NW;               // (nblk < 8: a wave may have none)
  auto tile_of = [&](int a) { return SWIGLU ? unit + a * p.pair_tiles : min(unit * T + a, p.ntiles - 1); };
  const char* gx = (const char*)p.xq + (size_t)__builtin_amdgcn_readfirstlane(slab) * p.G * 2 * X_HALF;
  const char* gw[T];
#pragma unroll
  for (int a = 0; a < T; ++a) gw[a] = (const char*)p.w + (size_t)tile_of(a) * p.nblk * 1152;
  const uint32_t lane16 = lane * 16, code_off = ((g >> 1) * 16 + c16) * 16 + (g & 1) * 8, sb_off = 1024 + c16 * 4;

  u32x4 x[2][2][MT];                                            // [group][k block][row tile]
  u32x2 cd[T][2];
  uint32_t sd[T], bd[T];
  f32x4 acc[T][MT];
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[a][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int LOADS = 4 * T + 4 * MT;                          // of a block: codes, scales, biases, x in the order of its use
  auto load = [&](int i, int l0, int l1) __attribute__((always_inline)) {
    const size_t blk = (size_t)(wave + NW * min(i, mine - 1));
    const char* xb = gx + blk * (4 * X_HALF);
#pragma unroll
    for (int l = l0; l < l1; ++l) {
      const char* w = gw[l % T] + blk * 1152;
      if (l < 2 * T) cd[l % T][l / T] = *(const u32x2*)(w + l / T * 512 + code_off);
      else if (l < 3 * T) sd[l % T] = *(const uint32_t*)(w + sb_off);
      else if (l < 4 * T) bd[l % T] = *(const uint32_t*)(w + sb_off + 64);
      else {
        const int j = l - 4 * T, sg = j / (2 * MT), m = j / 2 % MT, t = j & 1;
        x[sg][t][m] = *(const u32x4*)(xb + (sg * 2 + t) * X_HALF + m * 1024 + lane16);
      }
    }
  };
  uint32_t mask = 0x00780078u, magic = 0x41804180u;
  asm("" : "+v"(mask), "+v"(magic));
  auto unpack = [&](uint32_t q, int c) -> uint32_t {             // unpack_q4, a register at a time
    if constexpr (OFFS) return (c == 0 ? q << 3 : c == 1 ? q >> 1 : c == 2 ? q >> 5 : q >> 9) & mask | magic;
    else return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, ((q >> (4 * c)) & 0x000F000Fu) | 0x64006400u) - f16x2{(_Float16)1024.f, (_Float16)1024.f});
  };
  const uint32_t one = OFFS ? 0xC180C180u : 0x3C003C00u;         // -16 (bf16), 1 (f16)
  const u32x4 ones = {one, one, one, one};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // block i; the next one's loads go out between its products, a few at a time: in one piece they hold the wave up for what the CU's path takes of all
  f32x4 d[2][T], sx[2];
  float sc[2][T], bi[2][T];
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    sx[v] = zero;
#pragma unroll
    for (int a = 0; a < T; ++a) { d[v][a] = zero; sc[v][a] = bi[v][a] = 0.f; }
  }
  auto fold = [&](int v, int m, int sv) {
#pragma unroll
    for (int a = 0; a < T; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[a][m][r] = fmaf(bi[sv][a], sx[v][r], fmaf(sc[sv][a], d[v][a][r], acc[a][m][r]));
  };
  auto mult = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int sg = 0; sg < 2; ++sg) {
      u32x4 w[T][2];
#pragma unroll
      for (int a = 0; a < T; ++a) {
#pragma unroll
        for (int c = 0; c < 4; ++c) { w[a][0][c] = unpack(cd[a][sg].x, c); w[a][1][c] = unpack(cd[a][sg].y, c); }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int j = sg * MT + m, v = j & 1;
        __builtin_amdgcn_sched_barrier(0);
        sx[v] = mfma16<AT>(x[sg][0][m], ones, zero);
        sx[v] = mfma16<AT>(x[sg][1][m], ones, sx[v]);
#pragma unroll
        for (int a = 0; a < T; ++a) d[v][a] = mfma16<AT>(x[sg][0][m], w[a][0], OFFS ? sx[v] : zero);
#pragma unroll
        for (int a = 0; a < T; ++a) d[v][a] = mfma16<AT>(x[sg][1][m], w[a][1], d[v][a]);
        fold(v ^ 1, (m + MT - 1) % MT, j == 0 ? 1 : m == 0 ? 0 : sg);
        if (j == 0) {
#pragma unroll
          for (int a = 0; a < T; ++a)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              if constexpr (OFFS) {
                sc[u][a] = __uint_as_float(u ? sd[a] & 0xffff0000u : sd[a] << 16);
                bi[u][a] = __uint_as_float(u ? bd[a] & 0xffff0000u : bd[a] << 16) * -0.0625f;
              } else {
                sc[u][a] = (float)__builtin_bit_cast(f16, (unsigned short)(sd[a] >> (16 * u)));
                bi[u][a] = (float)__builtin_bit_cast(f16, (unsigned short)(bd[a] >> (16 * u)));
              }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // what this row tile leaves free takes the next block's
        if (m == 0) load(i + 1, T * sg, T * sg + T);
        if (j == 0) load(i + 1, 2 * T, 4 * T);
        load(i + 1, 4 * T + 2 * j, 4 * T + 2 * j + 2);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if (mine > 0) {
    load(0, 0, LOADS);
    for (int i = 0; i < mine; ++i) mult(i);
    fold((2 * MT - 1) & 1, MT - 1, 1);
  }

#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[((wave * T + a) * MT + m) * 64 + lane] = acc[a][m];
  // a wave's output tile (SwiGLU: pair): lane (c16, g) finishes rows 4 g .. 4 g + 3, column c16
  const int a_out = SWIGLU ? 0 : wave / MT, m_out = SWIGLU ? wave : wave % MT;
  const bool live = (SWIGLU ? wave < MT : wave < T * MT && unit * T + a_out < p.ntiles);
  const int n = tile_of(a_out) * 16 + c16, r0 = row0 + m_out * 16 + g * 4;
  float hres[4] = {0.f, 0.f, 0.f, 0.f};
  if (!SWIGLU && live && p.epi == EPI_RESID) {
#pragma unroll
    for (int r = 0; r < 4; ++r) hres[r] = (float)((const AT*)p.resid)[(size_t)min(r0 + r, p.M - 1) * p.ldo + n];
  }
  __syncthreads();
  if (!live) return;
  f32x4 y[SWIGLU ? 2 : 1];
#pragma unroll
  for (int v = 0; v < (SWIGLU ? 2 : 1); ++v) {
    const f32x4* src = red + ((a_out + v) * MT + m_out) * 64 + lane;
    y[v] = src[0];
#pragma unroll
    for (int k = 1; k < NW; ++k) y[v] += src[k * T * MT * 64];
  }
  AT* out = (AT*)p.out;
#pragma unroll 1
  for (int r = 0; r < 4; ++r) {                                  // (rolled: its branches stand once)
    const int row = r0 + r;
    if (row >= p.M) break;
    const float v = r == 0 ? y[0].x : r == 1 ? y[0].y : r == 2 ? y[0].z : y[0].w;
    if constexpr (SWIGLU) {
      const float up = r == 0 ? y[1].x : r == 1 ? y[1].y : r == 2 ? y[1].z : y[1].w;
      out[swiglu_at(p, row, n)] = silu16<AT>(v, up);
    } else {
      float z = (float)(AT)v;
      if (p.lora_t != nullptr) {
        for (int sl = 0; sl < 2; ++sl) {
          const int l0 = sl ? p.lora_row0_1 : p.lora_row0_0, ln = sl ? p.lora_n_1 : p.lora_n_0, rk = sl ? p.lora_rank_1 : p.lora_rank_0;
          const float* lb = sl ? p.lora_b1 : p.lora_b0;
          if (lb != nullptr && n >= l0 && n < l0 + ln) {
            const float t = (sl ? p.lora_scale_1 : p.lora_scale_0) * lora_dot(p.lora_t + (size_t)row * p.lora_t_ld + sl * (p.lora_t_ld / 2), lb + (n - l0), ln, rk);
            z = (float)(AT)(z + (float)(AT)t);
          }
        }
      }
      if (p.epi == EPI_STORE) out[(size_t)row * p.ldo + n] = (AT)z;
      else if (p.epi == EPI_STORE_F32) ((float*)p.out)[(size_t)row * p.ldo + n] = z;
      else ((AT*)p.resid)[(size_t)row * p.ldo + n] = (AT)((r == 0 ? hres[0] : r == 1 ? hres[1] : r == 2 ? hres[2] : hres[3]) + z);
    }
  }
}

struct Q4Plan { bool rows; int tn, mt, nslab, ksplit, ntu, ntiles, ngroups, nblk; size_t xq_bytes, sx_bytes, sxo_bytes, ws_bytes; };

thread_local int q4_force_mt = 0, q4_force_ks = 0;               // test hook: row tiles per workgroup, K slices (0: the plan's own)
thread_local int q4_force_rows = 0, q4_force_tn = 0;
thread_local bool q4_forced = false;                             // .. and whatever the width

// Narrow matrices: q4_rows_kernel or gemm_skinny.hip?  us, both with their preparation but without the norm launch of 4.7 that q4_prep_kernel saves, warm weights,
// here / there at 32, 64 and 128 rows: 7168 x 5120 11 / 15, 14 / 22, 26 / 30; 5120 x 5120 11 / 17, 15 / 22, 26 / 27; 4096 x 4096 10 / 15, 13 / 21, 15 / 23; 4096 x 6400 12 / 17,
// 16 / 24, 19 / 29; 8192 x 8192 15 / 22, 21 / 30, 38 / 45; 4096 x 10240 15 / 19, 22 / 29, 26 / 35; 4096 x 12288 17 / 22, 25 / 29, 29 / 38.  More than one round of workgroups: 5120 x 10240
// at 65 rows 36 / 33, 128 43 / 41; with a norm (to be added to the other side) or a SwiGLU 10240 x 5120 16 / 17, 25 / 25, 36 / 45; 10240 x 8192 22 / 22, 35 / 34, 51 / 59; 16128 x 8192
// 23 / 27, 36 / 44, 68 / 72; 16128 x 4096 15 / 18, 23 / 28, 41 / 38 (four rounds: behind by less than the norm); SwiGLU 14336 x 4096 15 / 19, 22 / 30, 39 / 41, 16128 x 8192 23 / 28, 36 / 43, 67 / 68.
// A longer K, one round: 4096 x 10240 15 / 19, 22 / 28, 27 / 35; 3072 x 11008 16 / 19, 24 / 27, 26 / 33; 4096 x 14336 20 / 22, 29 / 33, 35 / 43; 5120 x 17408 22 / 26, 34 / 40, in two rounds at
// 128 rows 67 / 62.  Few columns behind a long K leave CUs idle, which the other kernel splits K over (us at 17 / 64 / 128 rows; where the launch in front
// leaves x prepared the first is 4.8 less): 4096 x 22016 27 / 25, 40 / 38, 46 / 57, x 28672 33 / 29, 51 / 43, 58 / 68; 3072 x 17408 22 / 21, 33 / 31, 35 / 41, x 22016 26 / 23, 40 / 35, 43 / 49; 2048 x 10240 15 / 17, 22 / 23, 24 / 28,
// x 17408 21 / 20, 32 / 29, 35 / 34, x 22016 26 / 22, 40 / 32, 42 / 38; 1024 x 8704 13 / 15, 20 / 18, 21 / 24, x 17408 22 / 19, 33 / 22, 35 / 29.
// So: one round of workgroups up to K = 20480 or 6 N, and up to K = 8192 any number where a norm launch goes with the other kernel. A short K without a norm: the preparation is a launch of its own, 256 x 128 5.5 / 4.9, 6.0 / 5.4, 6.1 / 5.4;
// 512 x 256 5.8 / 5.7, 6.2 / 5.8, 6.3 / 5.8; 1024 x 512 6.0 / 6.5, 6.6 / 6.6, 6.7 / 6.7.  So from K = 512.
bool q4_rows_ahead(const LinearW& W, const GemvCall& c, size_t rows) {
  const long units = c.epi == EPI_SWIGLU ? c.pair_offset / 16 : (W.N / 16 + RT - 1) / RT, slabs = (long)((rows + 63) / 64);
  const bool one = units * slabs <= gemv_cu_count();
  return (W.K <= 8192 || (one && W.K <= std::max(20480, 6 * W.N))) && (c.pro == PRO_NORM || (W.K >= 512 && (c.epi == EPI_SWIGLU || one)));
}
bool q4_rows(const LinearW& W, const GemvCall& c) { return q4_force_rows > 0 || (!q4_forced && W.N / 16 < GEMM_Q4_MIN_TILES); }

// Column tiles a wave where K is not split (a column's sum is the same whatever it shares a wave with): four where their rounds of workgroups, each some 7/8 of one of five
// tiles, cost less.  us at 32 / 64 / 128 rows, five and four tiles: SwiGLU 28672 x 4096 25.5 / 32.5 / 61.5 and 23.3 / 28.6 / 52.4, 16384 x 4096 23.1 / 32.2 / 33.6 and
// 20.7 / 27.8 / 29.9, 44032 x 4096 46.8 / 61.4 / 91.7 and 40.2 / 51.8 / 79.2, logits 32000 x 4096 26.1 / 34.8 / 64.7 and 24.7 / 31.8 / 58.5, 128256 x 4096 100 / 136 / 228.5 and
// 92 / 124 / 227.1; a round more: SwiGLU 34816 x 5120 30.0 / 39.1 / 74.7 and 47.3 / 60.9 / 90.5, 19200 x 3072 at 128 rows 28.5 and 43.7, logits 151936 x 5120 128 / 169 / 309 and
// 135 / 174 / 323, 50304 x 3072 at 128 rows 81.3 and 90.5.
int q4_tiles(long groups4, long groups5) {
  if (q4_force_tn == 4 || q4_force_tn == 5) return q4_force_tn;
  const long cus = gemv_cu_count(), r4 = (groups4 + cus - 1) / cus, r5 = (groups5 + cus - 1) / cus;
  return 7 * r4 < 8 * r5 ? 4 : 5;
}

Q4Plan q4_plan(const LinearW& W, const GemvCall& c, size_t rows) {
  Q4Plan pl{};
  const bool sw = c.epi == EPI_SWIGLU;
  pl.ntiles = W.N / 16;
  pl.ntu = sw ? c.pair_offset / 16 : pl.ntiles;
  pl.nblk = W.K / 128;
  constexpr int TN = 5;
  const auto groups_of = [&](int tn) { return sw ? (pl.ntu + tn - 1) / tn : (pl.ntiles + TW * tn - 1) / (TW * tn); };
  pl.tn = TN;
  pl.ngroups = groups_of(TN);
  const int tiles = (int)((rows + 15) / 16);
  pl.nslab = (tiles + 3) / 4;
  pl.mt = std::max(2, (tiles + pl.nslab - 1) / pl.nslab);
  if (q4_force_mt > 0) { pl.mt = std::min(4, std::max(2, q4_force_mt)); pl.nslab = (tiles + pl.mt - 1) / pl.mt; }
  pl.rows = q4_rows(W, c);
  const double cus = gemv_cu_count(), step = 0.35 + 0.2 * pl.mt;
  double best = 1e30;
  if (pl.rows) { pl.ksplit = 1; pl.ngroups = sw ? pl.ntu : (pl.ntiles + RT - 1) / RT; }
  else for (int ks = 1; ks <= 8 && ks <= pl.nblk; ++ks) {
    const double rounds = std::ceil(pl.ngroups * pl.nslab * ks / cus), iters = ((pl.nblk + ks - 1) / ks + KW - 1) / KW;
    double t = rounds * (2.0 * iters * step + 5.0);
    if (ks > 1) t += 2.0 + 2.0 * ks * (double)pl.ngroups * TW * TN * pl.nslab * pl.mt * 1024 / 4.0e6;
    if (q4_force_ks > 0 ? ks == std::min(q4_force_ks, pl.nblk) : t < best) { best = t; pl.ksplit = ks; }
  }
  if (!pl.rows && pl.ksplit == 1 && q4_tiles(groups_of(4) * pl.nslab, pl.ngroups * pl.nslab) == 4) { pl.tn = 4; pl.ngroups = groups_of(4); }
  const size_t G = W.K / 64;
  pl.xq_bytes = (size_t)pl.nslab * G * 2 * pl.mt * 1024;
  pl.sx_bytes = pl.rows ? 0 : (pl.nslab * G * 16 * pl.mt * sizeof(float) + 255) & ~(size_t)255;
  pl.sxo_bytes = pl.rows ? 0 : pl.nslab * G * 256;
  pl.ws_bytes = pl.xq_bytes + pl.sx_bytes + pl.sxo_bytes + (pl.ksplit > 1 ? (size_t)pl.nslab * pl.ksplit * pl.ngroups * TW * TN * pl.mt * 1024 : 0);
  return pl;
}

template <typename AT, int MT, bool SW, int TN>
int q4_launch_k(const Q4Params& p, int grid, hipStream_t st) {
  auto kern = q4_kernel<AT, MT, SW, TN>;
  static std::atomic<bool> granted[64];
  MI_TRY(grant_lds((const void*)kern, Q4_LDS, granted));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * 64), Q4_LDS, st, p);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

template <typename AT, int TN>
int q4_launch_at(const Q4Params& p, int mt, bool sw, int grid, hipStream_t st) {
  switch (mt) {
    case 2: return sw ? q4_launch_k<AT, 2, true, TN>(p, grid, st) : q4_launch_k<AT, 2, false, TN>(p, grid, st);
    case 3: return sw ? q4_launch_k<AT, 3, true, TN>(p, grid, st) : q4_launch_k<AT, 3, false, TN>(p, grid, st);
    case 4: return sw ? q4_launch_k<AT, 4, true, TN>(p, grid, st) : q4_launch_k<AT, 4, false, TN>(p, grid, st);
  }
  return fail(MI_ERR_INVALID, "gemm_q4: 2..4 row tiles per workgroup");
}

template <typename AT>
int q4_rows_launch(const Q4Params& p, int mt, bool sw, int grid, hipStream_t st) {
  switch (mt) {
#define RK(MT) case MT: if (sw) hipLaunchKernelGGL((q4_rows_kernel<AT, MT, true>), dim3(grid), dim3(NW * 64), 0, st, p); \
                        else hipLaunchKernelGGL((q4_rows_kernel<AT, MT, false>), dim3(grid), dim3(NW * 64), 0, st, p); break;
    RK(2) RK(3) RK(4)
#undef RK
    default: return fail(MI_ERR_INVALID, "gemm_q4: 2..4 row tiles per workgroup");
  }
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace

// test hook: row tiles | .. << 3 | column tiles a wave << 7 (K not split; the field between is q4_kernel's fixed shape) | K slices << 11 | q4_rows_kernel << 15; 0 clears
void gemm_q4_force(int code) { q4_force_mt = code & 7; q4_force_tn = (code >> 7) & 15; q4_force_ks = (code >> 11) & 15; q4_force_rows = (code >> 15) & 1; q4_forced = code != 0; }

// The wide matrices, and the narrow ones of q4_rows_ahead.  Wide: us, 64 rows (32 rows), against gemm_skinny.hip's K over workgroups; with the preparation pass, which replaces a norm launch of
// 4.7 us in front of gate|up and the logits: 34816 x 5120 SwiGLU 42 (31) against 71 (40), 28672 x 4096 33 (25) against 40 (25), 151936 x 5120
// 172 (131) against 272 (149), 20480 x 5120 37 (27) against 42 (26).  A workgroup's head and tail are some 10 us, slices of K another 8: 5120 x 17408
// 42 (31) against 37 (26); few rows on short K: 50304 x 2048 45 (34) against 40 (22).
bool gemm_q4_supported(const LinearW& W, const GemvCall& c, size_t rows) {
  if (c.force_v1 || W.layout != 1 || c.rnd != RND_NONE || c.out32) return false;
  const bool q4 = ((W.wk == WK_Q4_BF16 && c.act == MI_BF16) || (W.wk == WK_Q4_F16 && c.act == MI_F16)) && W.group == 64 && W.K % 128 == 0;
  if (!q4 || rows < 17 || rows > 128 || c.ldx % 8 != 0) return false;
  if (c.epi == EPI_SWIGLU_GU8 || c.glu.kind != GLU_SILU || c.silu_cols > 0) return false;
  if (W.N % 16 != 0 || (c.epi == EPI_SWIGLU && c.pair_offset % 16 != 0)) return false;
  if (!q4_forced && (W.N / 16 < GEMM_Q4_MIN_TILES ? !q4_rows_ahead(W, c, rows) : (rows <= 32 && W.K < 3072))) return false;
  return (size_t)(W.N / 16) * (W.K / 128) * 1152 < ((size_t)1 << 32);          // (32-bit offsets of the LDS-DMA sources)
}

int gemm_q4_frag_mt(const LinearW& W, const GemvCall& c, size_t rows) {
  if (c.pro != PRO_NONE || !gemm_q4_supported(W, c, rows)) return 0;
  const Q4Plan pl = q4_plan(W, c, rows);
  return pl.rows ? pl.mt : 0;
}
size_t gemm_q4_ws_bytes(const LinearW& W, const GemvCall& c, size_t rows) { return q4_plan(W, c, rows).ws_bytes; }
int gemm_q4_ksplit(const LinearW& W, const GemvCall& c, size_t rows) { return q4_plan(W, c, rows).ksplit; }
int gemm_q4_groups(const LinearW& W, const GemvCall& c, size_t rows) {
  const Q4Plan pl = q4_plan(W, c, rows);
  return pl.ngroups * pl.nslab;
}

int launch_gemm_q4(const LinearW& W, const GemvCall& c, size_t rows, hipStream_t st, void* ws, unsigned* ctr) {
  if (!gemm_q4_supported(W, c, rows)) return fail(MI_ERR_INVALID, "gemm_q4: unsupported call");
  const Q4Plan pl = q4_plan(W, c, rows);
  if (c.x_frag > 0 && (!pl.rows || pl.mt != c.x_frag || c.pro != PRO_NONE)) return fail(MI_ERR_INVALID, "gemm_q4: x prepared for another call");
  if (c.x_frag == 0 && (ws == nullptr || (pl.ksplit > 1 && ctr == nullptr))) return fail(MI_ERR_INVALID, "gemm_q4: workspace missing");
  void* xq = ws;
  float* sx = (float*)((char*)ws + pl.xq_bytes);
  float* sxo = (float*)((char*)sx + pl.sx_bytes);
  if (c.x_frag == 0) {
    const void* nw = c.pro == PRO_NORM ? c.norm_w : nullptr;
    const dim3 grid(pl.nslab * pl.mt * 16, nw != nullptr ? 1 : (W.K + 2047) / 2048);
    (c.act == MI_BF16 ? q4_prep_launch<bf16> : q4_prep_launch<f16>)(c, grid, (int)rows, pl.mt, W.K, nw, xq, pl.rows ? nullptr : sx, sxo, st);
    MI_HIP(hipGetLastError());
  }
  Q4Params p{};
  p.xq = c.x_frag > 0 ? c.x : xq; p.sx = sx; p.sxo = sxo; p.M = (int)rows; p.G = W.K / 64; p.w = W.w;
  p.epi = c.epi; p.out = c.out; p.ldo = c.ldo; p.resid = c.resid; p.pair_tiles = c.epi == EPI_SWIGLU ? c.pair_offset / 16 : 0;
  if (c.out_frag > 0 && (c.epi != EPI_SWIGLU || c.out_frag != pl.mt || pl.ntu % 8 != 0)) return fail(MI_ERR_INVALID, "gemm_q4: fragment order for another call");
  p.out_frag = c.out_frag;
  p.ntu = pl.ntu; p.ntiles = pl.ntiles; p.nblk = pl.nblk; p.ksplit = pl.ksplit; p.nslab = pl.nslab; p.ngroups = pl.ngroups; p.nunits = pl.ngroups * pl.ksplit;
  p.ws = (float*)((char*)sxo + pl.sxo_bytes); p.ctr = ctr;
  p.lora_t = c.lora_t; p.lora_t_ld = c.lora_t_ld;
  p.lora_b0 = W.lora_b[0]; p.lora_b1 = W.lora_b[1];
  p.lora_row0_0 = W.lora_row0[0]; p.lora_n_0 = W.lora_n[0]; p.lora_rank_0 = W.lora_rank[0]; p.lora_scale_0 = W.lora_scale[0];
  p.lora_row0_1 = W.lora_row0[1]; p.lora_n_1 = W.lora_n[1]; p.lora_rank_1 = W.lora_rank[1]; p.lora_scale_1 = W.lora_scale[1];
  if (pl.rows) {
    p.wgs = pl.nslab > 1 ? (p.nunits + 7) / 8 * 8 * pl.nslab : p.nunits;
    // Read ahead only where a spare CU has at most four units to read for: what one asks for takes 0.4 us, a unit's round of blocks some 2.  Beyond, the launch waits for it: cold
    // matrices, 32 / 64 rows, us with and without, 160 units of 5120 x 5120 11.1 / 13.9 and 12.2 / 17.0, 192 of 6144 x 8192 16.2 / 21.2 and 16.6 / 23.7, 200 of 6400 x 5120
    // 12.3 / 16.1 and 12.4 / 17.4, 224 of 7168 x 5120 12.3 / 16.5 and 12.2 / 17.0, 240 of 7680 x 5120 20.8 / 23.0 and 12.4 / 17.2, 252 of 8064 x 5120 41 / 46 and 12.4 / 17.1.
    const int spare = gemv_cu_count() - p.wgs, grid = p.wgs + (spare * 4 >= p.nunits ? spare : 0);
    return c.act == MI_BF16 ? q4_rows_launch<bf16>(p, pl.mt, c.epi == EPI_SWIGLU, grid, st) : q4_rows_launch<f16>(p, pl.mt, c.epi == EPI_SWIGLU, grid, st);
  }
  const int blocks = pl.nslab > 1 ? (p.nunits + 7) / 8 * 8 * pl.nslab : p.nunits;
  const bool sw = c.epi == EPI_SWIGLU;
  if (pl.tn == 4) return c.act == MI_BF16 ? q4_launch_at<bf16, 4>(p, pl.mt, sw, blocks, st) : q4_launch_at<f16, 4>(p, pl.mt, sw, blocks, st);
  return c.act == MI_BF16 ? q4_launch_at<bf16, 5>(p, pl.mt, sw, blocks, st) : q4_launch_at<f16, 5>(p, pl.mt, sw, blocks, st);
}

}  // namespace mi
