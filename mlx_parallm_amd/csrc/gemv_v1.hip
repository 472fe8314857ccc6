// gemv_v1.hip -- generic weight-streaming skinny GEMM  y[M][N] = x[M][K] . W[N][K]^T  for M <= 8.
//
// Replaces nn.Linear / nn.QuantizedLinear (= x @ W.T / mx.quantized_matmul) at the call sites
// llama.py:64-67,93,143,160-165,250-252 and qwen3.py:37-40,63,115, with the neighbouring
// element-wise ops fused in: RMSNorm prologue (llama.py:175-177,205), residual add
// (llama.py:188,190), SwiGLU (llama.py:165), LoRALinear epilogue (mlx-lm, utils.py:742-744).
//
// This is the exact-fp32 VALU version that handles EVERY dtype combination (float32 /
// bfloat16 / float16 activations; dense or MLX-affine int4/int8 weights with scales in any
// of the three types).  The 16-bit hot configurations go through gemv_mfma.hip instead.
//
// Structure: one 256-thread workgroup = 4 waves; every wave owns PW row PAIRS of W and walks
// the whole K dimension; the 64 lanes split K in 16-byte pieces (coalesced 1 KiB per
// wave-instruction, weights go HBM -> VGPR directly, never through LDS); the activations are
// staged once per workgroup into LDS as fp32 in K-chunks of KC; fp32 accumulate; one
// butterfly reduction per row at the end.
#include <algorithm>

#include "kernels.h"

namespace mi {

int gemv_cu_count();      // gemv_mfma.hip

namespace {

constexpr int KC = 2048;  // K elements of x held in LDS at a time
constexpr int PW = 2;     // row pairs per wave
constexpr int NTHR = 256;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct GemvParams {
  const void* x; int ldx; int M;
  int rnd; int pro; const void* norm_w; float eps;
  const void* w; const void* scales; const void* biases;
  int N, K, group, layout;
  int epi; void* out; int ldo; void* resid; int pair_offset;
  Glu glu; int silu_cols;
  int out32;                   // GemvCall::out32
  int npairs;
  // LoRA
  const float* lora_t; int lora_t_ld;
  const float* lora_b0; const float* lora_b1;
  int lora_row0_0, lora_n_0, lora_rank_0; float lora_scale_0;
  int lora_row0_1, lora_n_1, lora_rank_1; float lora_scale_1;
  int lora_rnd;
};

// ---- 8 consecutive weights of one row, as fp32 -------------------------------------------
template <int WK>
__device__ __forceinline__ void load8(const GemvParams& p, int row, int kb, float (&o)[8]) {
  if constexpr (WK == WK_F32) {
    const float* base = (const float*)p.w + (size_t)row * p.K + kb;
    f32x4 a = __builtin_nontemporal_load((const f32x4*)base);
    f32x4 b = __builtin_nontemporal_load((const f32x4*)(base + 4));
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
  } else if constexpr (WK == WK_BF16) {
    const uint16_t* base = p.layout ? (const uint16_t*)((const char*)p.w + tiled_piece_dense16(row, kb, p.K))
                                    : (const uint16_t*)p.w + (size_t)row * p.K + kb;
    u32x4 v = __builtin_nontemporal_load((const u32x4*)base);
    o[0] = bf16lo(v.x); o[1] = bf16hi(v.x); o[2] = bf16lo(v.y); o[3] = bf16hi(v.y);
    o[4] = bf16lo(v.z); o[5] = bf16hi(v.z); o[6] = bf16lo(v.w); o[7] = bf16hi(v.w);
  } else if constexpr (WK == WK_F16) {
    const f16* base = p.layout ? (const f16*)((const char*)p.w + tiled_piece_dense16(row, kb, p.K))
                               : (const f16*)p.w + (size_t)row * p.K + kb;
    u32x4 v = __builtin_nontemporal_load((const u32x4*)base);
    const f16* h = (const f16*)&v;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (float)h[j];
  } else {
    constexpr int BITS = (WK >= WK_Q8_F32) ? 8 : 4;
    constexpr int SDT = (WK - 3) % 3;  // 0 f32, 1 bf16, 2 f16
    const int ng = p.K / p.group;
    const size_t gi = (size_t)row * ng + kb / p.group;
    float s, b;
    const char* blk = nullptr;
    if (BITS == 4 && SDT != 0 && p.layout) {       // tile-major int4 (repack.hip): scales live in the block
      blk = (const char*)p.w + tiled_block_q4(row, kb, p.K);
      const int so = tiled_q4_scale_off(row, kb);
      if constexpr (SDT == 1) { s = (float)*(const bf16*)(blk + so); b = (float)*(const bf16*)(blk + so + 64); }
      else { s = (float)*(const f16*)(blk + so); b = (float)*(const f16*)(blk + so + 64); }
    } else if (BITS == 8 && SDT != 0 && p.layout) {  // tile-major int8
      blk = (const char*)p.w + tiled_block_q8(row, kb, p.K);
      const int so = tiled_q8_scale_off(row);
      if constexpr (SDT == 1) { s = (float)*(const bf16*)(blk + so); b = (float)*(const bf16*)(blk + so + 32); }
      else { s = (float)*(const f16*)(blk + so); b = (float)*(const f16*)(blk + so + 32); }
    } else if constexpr (SDT == 0) { s = ((const float*)p.scales)[gi]; b = ((const float*)p.biases)[gi]; }
    else if constexpr (SDT == 1) { s = (float)((const bf16*)p.scales)[gi]; b = (float)((const bf16*)p.biases)[gi]; }
    else { s = (float)((const f16*)p.scales)[gi]; b = (float)((const f16*)p.biases)[gi]; }
    if constexpr (BITS == 4) {
      const uint32_t* base = blk ? (const uint32_t*)(blk + tiled_q4_code_off(row, kb))
                                 : (const uint32_t*)p.w + (size_t)row * (p.K / 8) + kb / 8;
      uint32_t v = __builtin_nontemporal_load(base);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = mul_add_unfused((float)((v >> (4 * j)) & 15u), s, b);
    } else {
      const uint32_t* base = blk ? (const uint32_t*)(blk + tiled_q8_code_off(row, kb))
                                 : (const uint32_t*)p.w + (size_t)row * (p.K / 4) + kb / 4;
      u32x2 v = __builtin_nontemporal_load((const u32x2*)base);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = mul_add_unfused((float)((v.x >> (8 * j)) & 255u), s, b);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[4 + j] = mul_add_unfused((float)((v.y >> (8 * j)) & 255u), s, b);
    }
  }
}

// LDS address (in floats) of x[m][kk] (kk inside the chunk): the 8 k's a lane needs for one
// 512-wide step are stored as two 16-byte halves [half][lane] so that each ds_read_b128 of a
// wave is 1 KiB contiguous (conflict free).
__device__ __forceinline__ int xs_addr(int m, int kk) {
  const int ks = kk >> 9, ln = (kk & 511) >> 3, half = (kk & 7) >> 2, j = kk & 3;
  return ((((m * (KC / 512) + ks) * 2 + half) * 64 + ln) << 2) + j;
}

// nn.silu(gate) * up, every op rounded to the activation dtype (llama.py:165), or another unit
template <typename AT>
__device__ __forceinline__ void finish_glu(const GemvParams& p, int m, int n, float gate, float up) {
  AT* out = (AT*)p.out;
  if (p.glu.kind != GLU_SILU) { out[(size_t)m * p.ldo + n] = store_act<AT>(glu_f(p.glu, gate, up), p.rnd); return; }
  const float g = to_f32(store_act<AT>(gate, p.rnd));
  const float u = to_f32(store_act<AT>(up, p.rnd));
  const float sig = to_f32(store_act<AT>(1.0f / (1.0f + expf(-g)), p.rnd));
  const float s = to_f32(store_act<AT>(g * sig, p.rnd));
  out[(size_t)m * p.ldo + n] = store_act<AT>(s * u, p.rnd);
}
// the other epilogues of y[m][n] = v
template <typename AT>
__device__ __forceinline__ void finish_one(const GemvParams& p, int m, int n, float v) {
  AT* out = (AT*)p.out;
  if (p.out32) {
    if (p.epi == EPI_RESID) { float* h32 = (float*)p.resid + (size_t)m * p.ldo + n; *h32 = *h32 + v; }
    else ((float*)p.out)[(size_t)m * p.ldo + n] = v;
    return;
  }
  float y = to_f32(store_act<AT>(silu_col(p.silu_cols, n, v), p.rnd));
  // LoRALinear: y + (scale * ((x A) B)).astype(x.dtype)
  if (p.lora_t != nullptr) {
#pragma unroll
    for (int sl = 0; sl < 2; ++sl) {
      const int row0 = sl ? p.lora_row0_1 : p.lora_row0_0;
      const int ln = sl ? p.lora_n_1 : p.lora_n_0;
      const int rk = sl ? p.lora_rank_1 : p.lora_rank_0;
      const float* lb = sl ? p.lora_b1 : p.lora_b0;
      if (lb != nullptr && n >= row0 && n < row0 + ln) {
        const float* t = p.lora_t + (size_t)m * p.lora_t_ld + sl * (p.lora_t_ld / 2);
        float z = 0.f;
        for (int j = 0; j < rk; ++j) z = fmaf(t[j], lb[(size_t)j * ln + (n - row0)], z);
        z = round_rt(z, p.lora_rnd);
        z = round_rt((sl ? p.lora_scale_1 : p.lora_scale_0) * z, p.lora_rnd);
        z = to_f32(store_act<AT>(z, p.rnd));
        y = to_f32(store_act<AT>(y + z, p.rnd));
      }
    }
  }
  if (p.epi == EPI_STORE) {
    out[(size_t)m * p.ldo + n] = from_f32<AT>(y);
  } else if (p.epi == EPI_STORE_F32) {
    ((float*)p.out)[(size_t)m * p.ldo + n] = y;
  } else {  // EPI_RESID
    AT* h = (AT*)p.resid;
    const float hv = to_f32(h[(size_t)m * p.ldo + n]);
    h[(size_t)m * p.ldo + n] = store_act<AT>(hv + y, p.rnd);
  }
}

template <typename AT, int WK, int MT>
__global__ __launch_bounds__(NTHR) void gemv_v1_kernel(GemvParams p) {
  extern __shared__ float smem[];
  float* xs = smem;                 // [MT][KC] permuted
  float* rs_sh = smem + MT * KC;    // [MT] rsqrt(mean(x^2)+eps)
  float* red = rs_sh + MT;          // [4][MT]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const AT* x = (const AT*)p.x;

  if (p.pro == PRO_NORM) {
    float ss[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) ss[m] = 0.f;
    for (int k = tid; k < p.K; k += NTHR) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        if (m < p.M) { float v = to_f32(x[(size_t)m * p.ldx + k]); ss[m] += v * v; }
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      float v = wave_sum(ss[m]);
      if (lane == 0) red[wave * MT + m] = v;
    }
    __syncthreads();
    if (tid < MT) {
      float v = red[tid] + red[MT + tid] + red[2 * MT + tid] + red[3 * MT + tid];
      rs_sh[tid] = 1.0f / sqrtf(v / (float)p.K + p.eps);
    }
    __syncthreads();
  }

  float acc[PW][2][MT];
#pragma unroll
  for (int a = 0; a < PW; ++a)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[a][r][m] = 0.f;

  int rows[PW][2];
  bool pvalid[PW];
#pragma unroll
  for (int a = 0; a < PW; ++a) {
    const int pair = (blockIdx.x * 4 + wave) * PW + a;
    pvalid[a] = pair < p.npairs;
    const int pp = pvalid[a] ? pair : 0;
    if (p.epi == EPI_SWIGLU) { rows[a][0] = pp; rows[a][1] = pp + p.pair_offset; }
    else { rows[a][0] = 2 * pp; rows[a][1] = min(2 * pp + 1, p.N - 1); }
  }

  const int nchunks = (p.K + KC - 1) / KC;
  for (int c = 0; c < nchunks; ++c) {
    if (c > 0) __syncthreads();
    // ---- stage x[:, c*KC : (c+1)*KC] (with the RMSNorm applied) into LDS as fp32
    for (int idx = tid * 4; idx < MT * KC; idx += NTHR * 4) {
      const int m = idx / KC, kk = idx % KC, k = c * KC + kk;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      if (m < p.M && k < p.K) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float t = to_f32(x[(size_t)m * p.ldx + k + j]);
          if (p.pro == PRO_NORM) {
            // w * cast_T(x32 * rsqrt(mean + eps))   
            AT xn = store_act<AT>(t * rs_sh[m], p.rnd);
            t = to_f32(store_act<AT>(to_f32(xn) * to_f32(((const AT*)p.norm_w)[k + j]), p.rnd));
          }
          v[j] = t;
        }
      }
      *(f32x4*)&xs[xs_addr(m, kk)] = f32x4{v[0], v[1], v[2], v[3]};
    }
    __syncthreads();

    const int ksteps = min(KC, p.K - c * KC);
    for (int ks = 0; ks * 512 < ksteps; ++ks) {
      const int kk = ks * 512 + lane * 8;
      const int kb = c * KC + kk;
      if (kb < p.K) {
        float w8[PW][2][8];
#pragma unroll
        for (int a = 0; a < PW; ++a)
#pragma unroll
          for (int r = 0; r < 2; ++r) load8<WK>(p, rows[a][r], kb, w8[a][r]);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int base = (((m * (KC / 512) + ks) * 2) * 64 + lane) << 2;
          const f32x4 x0 = *(const f32x4*)&xs[base];
          const f32x4 x1 = *(const f32x4*)&xs[base + 256];
#pragma unroll
          for (int a = 0; a < PW; ++a)
#pragma unroll
            for (int r = 0; r < 2; ++r) {
              float s = acc[a][r][m];
              s = fmaf(w8[a][r][0], x0.x, s); s = fmaf(w8[a][r][1], x0.y, s);
              s = fmaf(w8[a][r][2], x0.z, s); s = fmaf(w8[a][r][3], x0.w, s);
              s = fmaf(w8[a][r][4], x1.x, s); s = fmaf(w8[a][r][5], x1.y, s);
              s = fmaf(w8[a][r][6], x1.z, s); s = fmaf(w8[a][r][7], x1.w, s);
              acc[a][r][m] = s;
            }
        }
      }
    }
  }

  // ---- reduce over the 64 lanes; lane m finishes batch row m
#pragma unroll
  for (int a = 0; a < PW; ++a) {
    float mine[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float v = wave_sum(acc[a][r][m]);
        if (lane == m) mine[r] = v;
      }
    if (!pvalid[a] || lane >= p.M || lane >= MT) continue;
    const int m = lane;
    if (p.epi == EPI_SWIGLU) {
      finish_glu<AT>(p, m, rows[a][0], mine[0], mine[1]);
      continue;
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int n = rows[a][r];
      if (r == 1 && 2 * ((blockIdx.x * 4 + wave) * PW + a) + 1 >= p.N) continue;
      finish_one<AT>(p, m, n, mine[r]);
    }
  }
}

// the value of lane i ^ 4 (inside groups of 8: row_ror:4 for the upper four lanes, row_ror:12 for the lower)
__device__ __forceinline__ float xor4(float v) {
  const float up = __builtin_amdgcn_update_dpp(0.f, v, 0x124, 0xf, 0xa, false);
  return __builtin_amdgcn_update_dpp(up, v, 0x12C, 0xf, 0x5, false);
}
__device__ __forceinline__ float xor2_xor1(float v) {
  v += __builtin_amdgcn_update_dpp(0.f, v, 0x4E, 0xf, 0xf, false);    // quad_perm:[2,3,0,1]
  v += __builtin_amdgcn_update_dpp(0.f, v, 0xB1, 0xf, 0xf, false);    // quad_perm:[1,0,3,2]
  return v;
}

// Rows of at most 512 inputs.  In gemv_v1_kernel a wave spreads one row over its 64 lanes and every workgroup stages (and zero-fills)
// a 2048-wide image of x: at 64 inputs 8 of 64 lanes have work.  Here LG lanes hold a row (LG = 8, 16, 64), a wave takes 64 / LG of
// them at a time, and a lane keeps its 8 columns of x for every batch row in registers -- normed there, so nothing goes through LDS
// and no barrier stands in front of the weights.  int4, 64 inputs, 2 rows, float32 activations: 151936 outputs 74 -> 12 us, 192 outputs
// 9.8 -> 5.1 us (rocprof; an empty kernel is 4).  All sums are taken in gemv_v1_kernel's order: the results are the same bit for bit,
// whichever of the two an operand's alignment selects.
template <typename AT, int WK, int MT, int LG, bool GLU>
__global__ __launch_bounds__(NTHR) void gemv_short_kernel(GemvParams p) {
  constexpr int NR = GLU ? 2 : 1, RPW = 64 / LG, U = GLU || MT > 2 ? 2 : 4;
  const int tid = threadIdx.x, lane = tid & 63, grp = lane / LG, gl = lane % LG, k = gl * 8;
  const bool on = k < p.K;
  const AT* x = (const AT*)p.x;
  float xv[MT][8];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const AT* xr = x + (size_t)min(m, p.M - 1) * p.ldx + (on ? k : 0);
    alignas(16) AT e[8];
#pragma unroll
    for (int j = 0; j < (int)sizeof(AT) / 2; ++j) ((u32x4*)e)[j] = ((const u32x4*)xr)[j];
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[m][j] = on ? to_f32(e[j]) : 0.f;
  }
  auto group_sum = [&](float v) {                    // all-reduce over the LG lanes of a row
    if constexpr (LG == 8) return xor2_xor1(v + xor4(v));
    v = row16_sum(v);
    if constexpr (LG == 64) { v += __shfl_xor(v, 16); v += __shfl_xor(v, 32); }
    return v;
  };
  if (p.pro == PRO_NORM) {
    alignas(16) AT nw[8];
#pragma unroll
    for (int j = 0; j < (int)sizeof(AT) / 2; ++j) ((u32x4*)nw)[j] = ((const u32x4*)((const AT*)p.norm_w + (on ? k : 0)))[j];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma clang fp contract(off)                        // (the squares are rounded before they are added, there as here)
      // gemv_v1_kernel's order: thread t of 256 holds k = t (and t + 256), its wave_sum pairs k with k + 8, + 4, + 2, + 1 inside 16, the
      // four sixteens of 64 in pairs, the sixty-fours in sequence.  Here 64 columns are 8 lanes.
      float s[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] = xv[m][j] * xv[m][j];
      if constexpr (LG == 64)
        if (p.K > 256) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float far = __shfl_xor(xv[m][j], 32);
            s[j] = lane < 32 ? fmaf(far, far, s[j]) : 0.f;
          }
        }
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] += __builtin_amdgcn_update_dpp(0.f, s[j], 0xB1, 0xf, 0xf, false);     // quad_perm:[1,0,3,2]
      float t = ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
      t += __builtin_amdgcn_update_dpp(0.f, t, 0x4E, 0xf, 0xf, false);                                       // quad_perm:[2,3,0,1]
      t += xor4(t);
      if constexpr (LG == 16) t += __builtin_amdgcn_update_dpp(0.f, t, 0x128, 0xf, 0xf, false);              // row_ror:8
      if constexpr (LG == 64) {
        auto at = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, t), l)); };
        t = ((at(0) + at(8)) + at(16)) + at(24);
      }
      const float rs = 1.0f / sqrtf(t / (float)p.K + p.eps);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const AT xn = store_act<AT>(xv[m][j] * rs, p.rnd);
        xv[m][j] = on ? to_f32(store_act<AT>(to_f32(xn) * to_f32(nw[j]), p.rnd)) : 0.f;
      }
    }
  }
  const int items = GLU ? p.pair_offset : p.N, waves = gridDim.x * (NTHR / 64);
  for (int it0 = (blockIdx.x * (NTHR / 64) + (tid >> 6)) * RPW; it0 < items; it0 += waves * RPW * U) {      // (uniform per wave)
    float w8[U][NR][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = min(it0 + u * waves * RPW + grp, items - 1);
#pragma unroll
      for (int r = 0; r < NR; ++r) load8<WK>(p, it + r * p.pair_offset, on ? k : 0, w8[u][r]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = it0 + u * waves * RPW + grp;
      float mine[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        mine[r] = 0.f;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          float a = 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) a = fmaf(w8[u][r][j], xv[m][j], a);
          a = group_sum(on ? a : 0.f);                // (a lane past K read the row's first weights: 0 x inf is NaN)
          if (gl == m) mine[r] = a;
        }
      }
      if (it >= items || gl >= p.M || gl >= MT) continue;
      if constexpr (GLU) finish_glu<AT>(p, gl, it, mine[0], mine[1]);
      else finish_one<AT>(p, gl, it, mine[0]);
    }
  }
}

// t[m][slot][j] = round(sum_k xin[m][k] * A[k][j]); xin = (normed) x, same prologue as above.
// What bounds it is round trips to L2, so a workgroup is 8 waves and takes 2048 k at a time with all loads in flight; four lanes read a row of A (16 ranks), a
// wave one KiB -- a lane that reads whole rows, 64 bytes apart, costs the CU's path four times the cycles.  x goes through LDS, normalised once.
// 64 rows x 5120 at rank 16, both slots: 23.5 us (four waves, a row of A per lane) -> 11.8.
constexpr int LD_NTHR = 512, LD_KC = 2048;
// VEC: ranks in fours.  (NORM and VEC are forms: asked inside, they make a branch of every load)
template <typename AT, bool NORM, bool VEC>
__global__ __launch_bounds__(LD_NTHR) void lora_down_kernel(GemvParams p, const float* a0, const float* a1,
                                                            float* t, int t_ld) {
  constexpr int NW = LD_NTHR / 64, ROWS = LD_NTHR / 4, U = LD_KC / ROWS, XU = LD_KC / LD_NTHR;
  __shared__ float red[NW], red16[NW][16], xs[LD_KC];
  const int m = blockIdx.x, slot = blockIdx.y;
  const float* A = slot ? a1 : a0;
  const int rk = slot ? p.lora_rank_1 : p.lora_rank_0;
  if (A == nullptr) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = tid & 3;
  const AT* x = (const AT*)p.x + (size_t)m * p.ldx;
  float rs = 1.0f;
  if constexpr (NORM) {
    float ss = 0.f;
    for (int k0 = tid; k0 < p.K; k0 += 8 * LD_NTHR) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = to_f32(x[min(k0 + u * LD_NTHR, p.K - 1)]);
#pragma unroll
      for (int u = 0; u < 8; ++u) ss = k0 + u * LD_NTHR < p.K ? fmaf(v[u], v[u], ss) : ss;
    }
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) ss += red[w];
    rs = 1.0f / sqrtf(ss / (float)p.K + p.eps);
  }
  for (int j0 = 0; j0 < rk; j0 += 16) {
    const int jq = j0 + 4 * q;
    float s[4][4];                                               // four chains per column
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) s[u][j] = 0.f;
    for (int c0 = 0; c0 < p.K; c0 += LD_KC) {
      const int n = min(LD_KC, p.K - c0);
      float4 a4[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float* ar = A + (size_t)(c0 + min((tid >> 2) + u * ROWS, n - 1)) * rk;
        if constexpr (VEC) a4[u] = *(const float4*)(ar + (jq < rk ? jq : 0));
        else a4[u] = {ar[min(jq, rk - 1)], ar[min(jq + 1, rk - 1)], ar[min(jq + 2, rk - 1)], ar[min(jq + 3, rk - 1)]};
      }
      float v[XU], nw[XU];
#pragma unroll
      for (int u = 0; u < XU; ++u) {
        const int k = c0 + min(tid + u * LD_NTHR, n - 1);
        v[u] = to_f32(x[k]);
        nw[u] = NORM ? to_f32(((const AT*)p.norm_w)[k]) : 1.0f;
      }
      __syncthreads();                                           // (the last chunk has been read)
#pragma unroll
      for (int u = 0; u < XU; ++u) {
        if constexpr (NORM) {
          const AT xn = store_act<AT>(v[u] * rs, p.rnd);
          v[u] = to_f32(store_act<AT>(to_f32(xn) * nw[u], p.rnd));
        }
        xs[tid + u * LD_NTHR] = tid + u * LD_NTHR < n ? v[u] : 0.f;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = (tid >> 2) + u * ROWS;
        const bool on = i < n;                                   // (xs is zero there, but A may be infinite)
        const float xv = xs[i];
        s[u & 3][0] = fmaf(xv, on ? a4[u].x : 0.f, s[u & 3][0]);
        s[u & 3][1] = fmaf(xv, on ? a4[u].y : 0.f, s[u & 3][1]);
        s[u & 3][2] = fmaf(xv, on ? a4[u].z : 0.f, s[u & 3][2]);
        s[u & 3][3] = fmaf(xv, on ? a4[u].w : 0.f, s[u & 3][3]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {                                // (columns past the rank: of others, never stored)
      float w = (s[0][j] + s[1][j]) + (s[2][j] + s[3][j]);
#pragma unroll
      for (int o = 4; o < 64; o <<= 1) w += __shfl_xor(w, o, 64);
      if (lane < 4) red16[wave][4 * q + j] = w;
    }
    __syncthreads();
    if (tid < 16 && j0 + tid < rk) {
      float w = 0.f;
#pragma unroll
      for (int i = 0; i < NW; ++i) w += red16[i][tid];
      t[(size_t)m * t_ld + slot * (t_ld / 2) + j0 + tid] = round_rt(w, p.lora_rnd);
    }
  }
}

// y[m][n] = T(y[m][n] + T(scale * sum_j t[m][slot][j] * B[j][n - row0]))  for the adapted column ranges: the LoRA term
// of the GEMV epilogues, applied after a tile GEMM has stored y = T(x W^T) (prefill)
template <typename AT>
__global__ __launch_bounds__(256) void lora_up_add_kernel(GemvParams p, const float* t, int t_ld, AT* y, int ldy) {
  const int m = blockIdx.x;
#pragma unroll
  for (int sl = 0; sl < 2; ++sl) {
    const float* lb = sl ? p.lora_b1 : p.lora_b0;
    if (lb == nullptr) continue;
    const int r0 = sl ? p.lora_row0_1 : p.lora_row0_0;
    const int ln = sl ? p.lora_n_1 : p.lora_n_0;
    const int rk = sl ? p.lora_rank_1 : p.lora_rank_0;
    const float sc = sl ? p.lora_scale_1 : p.lora_scale_0;
    const float* tt = t + (size_t)m * t_ld + sl * (t_ld / 2);
    for (int n = threadIdx.x; n < ln; n += 256) {
      float z = lora_dot(tt, lb + n, ln, rk);
      z = sc * z;
      AT* o = y + (size_t)m * ldy + r0 + n;
      if constexpr (sizeof(AT) == 4) *o = round_rt((float)*o + round_rt(z, p.rnd), p.rnd);   // float32 storage, logical rounding (layer 0 of the PagedKVCache mode)
      else *o = (AT)((float)*o + (float)(AT)z);
    }
  }
}

template <typename AT, int WK, int MT>
int launch_short(const GemvParams& p, hipStream_t st) {
  const bool glu = p.epi == EPI_SWIGLU;
  const int lg = p.K <= 64 ? 8 : p.K <= 128 ? 16 : 64;
  const int items = glu ? p.pair_offset : p.N;
  // More rows than the grid holds are looped over.  Four workgroups per CU: that many of the largest instantiation (MT = 8: 105 to 125
  // registers) run at once, and each further one loads and norms x again.  1024 against 2048 workgroups, us: int4, 64 inputs, 151936 outputs,
  // float32 rows 8.8 / 10.2 (1 row), 11.2 / 14.8 (3), 17.8 / 25.3 (8); float32 weights, 512 inputs, 16384 outputs 10.2 / 14.9, 12.2 / 15.7, 18.3 /
  // 27.0.  Eight where the small instantiation has four rounds of loads for all of them: int4, 256 inputs, 151936 outputs 30.8 / 27.2 (1 row).
  const int per_wg = 4 * (64 / lg), per_cu = MT == 2 && items >= 4 * (8 * gemv_cu_count()) * per_wg * (glu ? 2 : 4) ? 8 : 4;
  const int nwg = std::min(per_cu * gemv_cu_count(), (items + per_wg - 1) / per_wg);
  auto go = [&](auto kern) -> int {
    hipLaunchKernelGGL(kern, dim3(nwg), dim3(NTHR), 0, st, p);
    MI_HIP(hipGetLastError());
    return MI_OK;
  };
#define GO(LG) return glu ? go(gemv_short_kernel<AT, WK, MT, LG, true>) : go(gemv_short_kernel<AT, WK, MT, LG, false>)
  if (lg == 8) GO(8);
  if (lg == 16) GO(16);
  GO(64);
#undef GO
}

template <typename AT, int WK>
int launch_mt(const GemvParams& p, hipStream_t st) {
  // short rows: x and the norm weights are read 16 bytes at a time there
  const bool al = ((uintptr_t)p.x | (uintptr_t)(p.pro == PRO_NORM ? p.norm_w : nullptr)) % 16 == 0 && (size_t)p.ldx * sizeof(AT) % 16 == 0;
  if (p.K <= 512 && al) {
    if (p.M <= 2) return launch_short<AT, WK, 2>(p, st);
    if (p.M <= 4) return launch_short<AT, WK, 4>(p, st);
    return launch_short<AT, WK, 8>(p, st);
  }
  const int nwg = (p.npairs + 4 * PW - 1) / (4 * PW);
  auto go = [&](auto kern, int MT) -> int {
    const size_t lds = (size_t)(MT * KC + MT + 4 * MT) * sizeof(float);
    static thread_local const void* configured[4] = {nullptr, nullptr, nullptr, nullptr};
    (void)configured;
    MI_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(nwg), dim3(NTHR), lds, st, p);
    MI_HIP(hipGetLastError());
    return MI_OK;
  };
  if (p.M <= 1) return go(gemv_v1_kernel<AT, WK, 1>, 1);
  if (p.M <= 4) return go(gemv_v1_kernel<AT, WK, 4>, 4);
  return go(gemv_v1_kernel<AT, WK, 8>, 8);
}

template <typename AT>
int launch_wk(int wk, const GemvParams& p, hipStream_t st) {
  constexpr bool F32A = sizeof(AT) == 4;
  switch (wk) {
    case WK_F32: if constexpr (F32A) return launch_mt<AT, WK_F32>(p, st); break;
    case WK_BF16: if constexpr (F32A || std::is_same<AT, bf16>::value) return launch_mt<AT, WK_BF16>(p, st); break;
    case WK_F16: if constexpr (F32A || std::is_same<AT, f16>::value) return launch_mt<AT, WK_F16>(p, st); break;
    case WK_Q4_F32: if constexpr (F32A) return launch_mt<AT, WK_Q4_F32>(p, st); break;
    case WK_Q8_F32: if constexpr (F32A) return launch_mt<AT, WK_Q8_F32>(p, st); break;
    case WK_Q4_BF16: if constexpr (F32A || std::is_same<AT, bf16>::value) return launch_mt<AT, WK_Q4_BF16>(p, st); break;
    case WK_Q8_BF16: if constexpr (F32A || std::is_same<AT, bf16>::value) return launch_mt<AT, WK_Q8_BF16>(p, st); break;
    case WK_Q4_F16: if constexpr (F32A || std::is_same<AT, f16>::value) return launch_mt<AT, WK_Q4_F16>(p, st); break;
    case WK_Q8_F16: if constexpr (F32A || std::is_same<AT, f16>::value) return launch_mt<AT, WK_Q8_F16>(p, st); break;
  }
  return fail(MI_ERR_UNSUPPORTED, "gemv: weight kind / activation dtype combination not supported");
}

GemvParams make_params(const LinearW& W, const GemvCall& c) {
  GemvParams p{};
  p.x = c.x; p.ldx = c.ldx; p.M = c.M; p.rnd = c.rnd; p.pro = c.pro; p.norm_w = c.norm_w; p.eps = c.eps;
  p.w = W.w; p.scales = W.scales; p.biases = W.biases; p.N = W.N; p.K = W.K; p.group = W.group; p.layout = W.layout;
  p.epi = c.epi; p.out = c.out; p.ldo = c.ldo; p.resid = c.resid; p.pair_offset = c.pair_offset;
  p.glu = c.glu; p.silu_cols = c.silu_cols;
  p.out32 = c.out32;
  p.npairs = (c.epi == EPI_SWIGLU) ? c.pair_offset : (W.N + 1) / 2;
  p.lora_t = c.lora_t; p.lora_t_ld = c.lora_t_ld;
  p.lora_b0 = W.lora_b[0]; p.lora_b1 = W.lora_b[1];
  p.lora_row0_0 = W.lora_row0[0]; p.lora_n_0 = W.lora_n[0]; p.lora_rank_0 = W.lora_rank[0]; p.lora_scale_0 = W.lora_scale[0];
  p.lora_row0_1 = W.lora_row0[1]; p.lora_n_1 = W.lora_n[1]; p.lora_rank_1 = W.lora_rank[1]; p.lora_scale_1 = W.lora_scale[1];
  p.lora_rnd = RND_NONE;
  return p;
}

}  // namespace

int launch_gemv_v1(const LinearW& W, const GemvCall& c, hipStream_t st) {
  if (c.M < 1 || c.M > 8) return fail(MI_ERR_INVALID, "gemv_v1: M must be in [1,8]");
  if (W.K % 8 != 0) return fail(MI_ERR_UNSUPPORTED, "gemv: K must be a multiple of 8");
  if (wk_is_quant(W.wk) && (W.group % 8 != 0 || W.K % W.group != 0))
    return fail(MI_ERR_UNSUPPORTED, "gemv: bad quantisation group size");
  if (c.epi == EPI_SWIGLU && c.pair_offset * 2 != W.N) return fail(MI_ERR_INVALID, "gemv: swiglu needs N = 2*pair_offset");
  GemvParams p = make_params(W, c);
  switch (c.act) {
    case MI_F32: return launch_wk<float>(W.wk, p, st);
    case MI_BF16: return launch_wk<bf16>(W.wk, p, st);
    case MI_F16: return launch_wk<f16>(W.wk, p, st);
  }
  return fail(MI_ERR_INVALID, "gemv: bad activation dtype");
}

template <typename AT>
static void lora_down_at(const GemvParams& p, const LinearW& W, float* t, int t_ld, hipStream_t st) {
  const dim3 grid(p.M, 2), block(LD_NTHR);
  const bool vec = (W.lora_rank[0] | W.lora_rank[1]) % 4 == 0;
#define LD_GO(N, V) hipLaunchKernelGGL((lora_down_kernel<AT, N, V>), grid, block, 0, st, p, W.lora_a[0], W.lora_a[1], t, t_ld)
  if (p.pro == PRO_NORM) { if (vec) LD_GO(true, true); else LD_GO(true, false); }
  else { if (vec) LD_GO(false, true); else LD_GO(false, false); }
#undef LD_GO
}

int launch_lora_down(const LinearW& W, const GemvCall& c, float* t, int t_ld, hipStream_t st) {
  const GemvParams p = make_params(W, c);
  switch (c.act) {
    case MI_F32: lora_down_at<float>(p, W, t, t_ld, st); break;
    case MI_BF16: lora_down_at<bf16>(p, W, t, t_ld, st); break;
    case MI_F16: lora_down_at<f16>(p, W, t, t_ld, st); break;
    default: return fail(MI_ERR_INVALID, "lora_down: bad activation dtype");
  }
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// c.out ([rows][ldo], EPI_STORE) += the LoRA term, rows = c.M, from t = launch_lora_down's output
int launch_lora_up_add(const LinearW& W, const GemvCall& c, const float* t, int t_ld, hipStream_t st) {
  if (c.epi != EPI_STORE) return fail(MI_ERR_UNSUPPORTED, "lora_up_add: plain store epilogue only");
  GemvParams p = make_params(W, c);
  const dim3 grid(c.M), block(256);
  switch (c.act) {
    case MI_BF16: hipLaunchKernelGGL(lora_up_add_kernel<bf16>, grid, block, 0, st, p, t, t_ld, (bf16*)c.out, c.ldo); break;
    case MI_F16: hipLaunchKernelGGL(lora_up_add_kernel<f16>, grid, block, 0, st, p, t, t_ld, (f16*)c.out, c.ldo); break;
    case MI_F32: hipLaunchKernelGGL(lora_up_add_kernel<float>, grid, block, 0, st, p, t, t_ld, (float*)c.out, c.ldo); break;
    default: return fail(MI_ERR_UNSUPPORTED, "lora_up_add: bad activation dtype");
  }
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
