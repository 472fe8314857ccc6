// repack.hip -- one-time conversion of a weight matrix from the checkpoint's row-major layout
// (W[N][K], MLX / safetensors order) to the tile-major layout the streaming kernels read.
//
// Why: a wave of the skinny-GEMM kernel consumes a 16-row x 32-k (dense 16-bit) or 16-row x 128-k
// (int4) block per load instruction.  Row-major, that block is 16 separate 64-byte pieces 2*K bytes
// apart; tile-major it is ONE contiguous KiB, and a workgroup's whole K sweep over its rows is one
// sequential stream -- measured +10..14 % on the decode GEMVs (4096 x 4096 .. 28672 x 4096, batch 8).
//
// Layouts (N % 16 == 0):
//   dense 16-bit: block (i = row/16, j = k/32) at ((i * K/32 + j) * 1024) bytes; inside, lane
//                 l = g*16 + r (r = row%16, g = (k%32)/8) owns bytes [16 l, 16 l + 16) = W[16i+r][32j+8g .. +8].
//   int4 (g64):   block (i, j = k/128) at ((i * K/128 + j) * 1152) bytes:
//                 [0,1024)    codes: lane l = g*16 + r owns the 4 packed dwords 4g..4g+3 of row r's 16
//                 [1024,1088) scales: row r -> 2 x 16-bit (quantisation groups 2j, 2j+1)
//                 [1088,1152) biases: same shape.
//   int8 (g64):   block (i, j = k/64) at ((i * K/64 + j) * 1088) bytes:
//                 [0,1024)    codes: lane l = g*16 + r owns the 16 codes W[16i+r][64j + 16g .. +16) (4 packed dwords)
//                 [1024,1056) scales: row r -> one 16-bit value;  [1056,1088) biases.
#include "kernels.h"

namespace mi {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__global__ void repack_dense16_kernel(const uint16_t* src, uint16_t* dst, int N, int K) {
  const size_t pieces = (size_t)N * (K / 8);
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < pieces; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t blk = idx >> 6;
    const int lane = (int)(idx & 63), r = lane & 15, g = lane >> 4;
    const size_t i = blk / (K / 32), j = blk % (K / 32);
    const u32x4 v = *(const u32x4*)(src + (i * 16 + r) * (size_t)K + j * 32 + g * 8);
    *(u32x4*)(dst + idx * 8) = v;
  }
}

__global__ void repack_q4_kernel(const uint32_t* codes, const uint16_t* scales, const uint16_t* biases, uint8_t* dst,
                                 int N, int K) {
  const int nb = K / 128;
  const size_t blocks = (size_t)(N / 16) * nb;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < blocks * 64; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t blk = idx >> 6;
    const int lane = (int)(idx & 63), r = lane & 15, g = lane >> 4;
    const size_t i = blk / nb, j = blk % nb;
    const size_t row = i * 16 + r;
    uint8_t* base = dst + blk * 1152;
    *(u32x4*)(base + lane * 16) = *(const u32x4*)(codes + row * (K / 8) + j * 16 + g * 4);
    if (g == 0) {
      *(uint32_t*)(base + 1024 + r * 4) = *(const uint32_t*)(scales + row * (K / 64) + j * 2);
      *(uint32_t*)(base + 1088 + r * 4) = *(const uint32_t*)(biases + row * (K / 64) + j * 2);
    }
  }
}

__global__ void repack_q8_kernel(const uint32_t* codes, const uint16_t* scales, const uint16_t* biases, uint8_t* dst,
                                 int N, int K) {
  const int nb = K / 64;
  const size_t blocks = (size_t)(N / 16) * nb;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < blocks * 64; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t blk = idx >> 6;
    const int lane = (int)(idx & 63), r = lane & 15, g = lane >> 4;
    const size_t i = blk / nb, j = blk % nb;
    const size_t row = i * 16 + r;
    uint8_t* base = dst + blk * 1088;
    *(u32x4*)(base + lane * 16) = *(const u32x4*)(codes + row * (K / 4) + j * 16 + g * 4);
    if (g == 0) {
      *(uint16_t*)(base + 1024 + r * 2) = scales[row * (K / 64) + j];
      *(uint16_t*)(base + 1056 + r * 2) = biases[row * (K / 64) + j];
    }
  }
}

// int4 tile-major -> dense 16-bit tile-major [hi | lo] with K' = 2K (the prefill GEMM's operand for quantised
// weights): w = scale * q + bias in float32 (as the oracle dequantises), hi = T(w), lo = T(w - hi), so that
// x . hi + x . lo reproduces x . w to 2^-17 relative -- below the accumulation-order noise of any fp32 GEMM.
// One thread per destination 16-byte piece of the hi half (coalesced writes; the codes are read once).
template <typename T>
__global__ void dequant_q4_hilo_kernel(const uint8_t* src, T* dst, int N, int K) {
  const size_t pieces = (size_t)N * (K / 8);
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < pieces; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t blk = idx >> 6;
    const int lane = (int)(idx & 63), r = lane & 15, g = lane >> 4;
    const size_t i = blk / (K / 32), j = blk % (K / 32);
    const size_t row = i * 16 + r;
    const int k = (int)j * 32 + g * 8;
    const uint8_t* qb = src + tiled_block_q4(row, k, K);
    const uint32_t codes = *(const uint32_t*)(qb + tiled_q4_code_off(row, k));
    const float s = (float)*(const T*)(qb + tiled_q4_scale_off(row, k));
    const float b = (float)*(const T*)(qb + tiled_q4_scale_off(row, k) + 64);
    T hi[8], lo[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float w = mul_add_unfused(s, (float)((codes >> (4 * e)) & 15u), b);
      hi[e] = (T)w;
      lo[e] = (T)(w - (float)hi[e]);
    }
    const size_t kb2 = (size_t)(2 * K) / 32;                       // 32-k blocks per row tile in the destination
    T* dh = dst + ((i * kb2 + j) * 64 + lane) * 8;
    T* dl = dst + ((i * kb2 + (size_t)(K / 32) + j) * 64 + lane) * 8;
    *(u32x4*)dh = *(const u32x4*)hi;
    *(u32x4*)dl = *(const u32x4*)lo;
  }
}

// the same for tile-major int8
template <typename T>
__global__ void dequant_q8_hilo_kernel(const uint8_t* src, T* dst, int N, int K) {
  const size_t pieces = (size_t)N * (K / 8);
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < pieces; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t blk = idx >> 6;
    const int lane = (int)(idx & 63), r = lane & 15, g = lane >> 4;
    const size_t i = blk / (K / 32), j = blk % (K / 32);
    const size_t row = i * 16 + r;
    const int k = (int)j * 32 + g * 8;
    const uint8_t* qb = src + tiled_block_q8(row, k, K);
    const uint8_t* cp = qb + tiled_q8_code_off(row, k);
    const uint32_t c0 = *(const uint32_t*)cp, c1 = *(const uint32_t*)(cp + 4);
    const float s = (float)*(const T*)(qb + tiled_q8_scale_off(row));
    const float b = (float)*(const T*)(qb + tiled_q8_scale_off(row) + 32);
    T hi[8], lo[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t q = ((e < 4 ? c0 : c1) >> (8 * (e & 3))) & 255u;
      const float w = mul_add_unfused(s, (float)q, b);
      hi[e] = (T)w;
      lo[e] = (T)(w - (float)hi[e]);
    }
    const size_t kb2 = (size_t)(2 * K) / 32;
    T* dh = dst + ((i * kb2 + j) * 64 + lane) * 8;
    T* dl = dst + ((i * kb2 + (size_t)(K / 32) + j) * 64 + lane) * 8;
    *(u32x4*)dh = *(const u32x4*)hi;
    *(u32x4*)dl = *(const u32x4*)lo;
  }
}

// tile-major int4 / int8 -> the operands of the tile GEMM on codes (gemm_prefill.hip: gemm_codes256_kernel):
//   codes  [N/16][K/32] KiB blocks of 16-bit integers (of T: -128..127 are exact in bf16 and f16), code - 8 (int4) or - 128 (int8), dense layout
//   wb     [N/16][kb/32] KiB blocks of bf16: what meets the group sums of x, column c = term * K/64 + group: a part (codes16_bias_part) of
//          bias + 8 s (128 s); zeros up to kb
//   sc     [N/16][K/64][16] float32: the scales
// Bound by its writes (2 bytes a code, half of the [hi | lo] copy's).  28672 x 4096: 52 us with the scales and biases, 6.2 TB/s
// the scales and biases of a row tile; bias: [K/64][16] of LDS
template <typename T, int BITS>
__device__ __forceinline__ void codes16_side(const uint8_t* src, uint16_t* wb, float* sc, int K, int kb, int big_first, size_t tile, float* bias) {
  constexpr int MID = BITS == 4 ? 8 : 128;
  const int G = K / 64, tid = threadIdx.x;
  for (int o = tid; o < G * 16; o += 256) {
    const int grp = o >> 4, r = o & 15;
    const T* sb = BITS == 4 ? (const T*)(src + (tile * (G / 2) + (grp >> 1)) * 1152 + 1024 + r * 4 + (grp & 1) * 2)
                            : (const T*)(src + (tile * G + grp) * 1088 + 1024 + r * 2);
    const float s = (float)sb[0];
    sc[tile * G * 16 + o] = s;
    bias[o] = fmaf((float)MID, s, (float)sb[BITS == 4 ? 32 : 16]);
  }
  __syncthreads();
  for (int o = tid; o < kb * 2; o += 256) {                         // (kb / 32 blocks of 64 pieces)
    const int r = o & 15, c0 = (o >> 6) * 32 + ((o >> 4) & 3) * 8;
    int term = c0 / G, grp = c0 - term * G;
    __bf16 v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = term < CODES16_TERMS ? (__bf16)bf16_part(bias[grp * 16 + r], codes16_bias_part(big_first ? CODES16_TERMS - 1 - term : term)) : (__bf16)0.f;
      if (++grp == G) { grp = 0; ++term; }
    }
    *(u32x4*)(wb + (tile * kb * 2 + o) * 8) = *(const u32x4*)v;
  }
}

// blockIdx.y = row tile; workgroup 0 of a tile its scales and biases, the others a block of 1024 bytes of codes a wave: 16 bytes a lane in, 32 (16) codes
// out as pieces of 8 k.
template <typename T, int BITS>
__global__ __launch_bounds__(256) void codes16_kernel(const uint8_t* src, T* codes, uint16_t* wb, float* sc, int K, int kb, int big_first) {
  constexpr int KB = BITS == 4 ? 128 : 64, BYTES = BITS == 4 ? 1152 : 1088, MID = BITS == 4 ? 8 : 128;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, nb = K / KB;
  const size_t tile = blockIdx.y;
  extern __shared__ float bias[];
  if (blockIdx.x == 0) { codes16_side<T, BITS>(src, wb, sc, K, kb, big_first, tile, bias); return; }
  for (int j = (blockIdx.x - 1) * 4 + (threadIdx.x >> 6); j < nb; j += (gridDim.x - 1) * 4) {
    const u32x4 q = *(const u32x4*)(src + (tile * nb + j) * BYTES + lane * 16);
    T* out = codes + tile * 16 * (size_t)K;
#pragma unroll
    for (int e = 0; e < (BITS == 4 ? 4 : 2); ++e) {
      T v[8];
      int kb32, slot;                                               // 32-k block of the tile, piece in it
      if constexpr (BITS == 4) {                                    // dword 4 g + e of the row's 16
        const uint32_t lo = q[e] & 0x0f0f0f0fu, hi = (q[e] >> 4) & 0x0f0f0f0fu;
#pragma unroll
        for (int i = 0; i < 4; ++i) { v[2 * i] = (T)((float)((lo >> (8 * i)) & 255u) - MID); v[2 * i + 1] = (T)((float)((hi >> (8 * i)) & 255u) - MID); }
        kb32 = 4 * j + g; slot = e;
      } else {                                                      // codes 16 g + 8 e .. + 8 of the row's 64
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (T)((float)((q[2 * e + (i >> 2)] >> (8 * (i & 3))) & 255u) - MID);
        kb32 = 2 * j + (g >> 1); slot = 2 * (g & 1) + e;
      }
      *(u32x4*)(out + ((size_t)kb32 * 64 + slot * 16 + r) * 8) = *(const u32x4*)v;
    }
  }
}

}  // namespace

int codes16_bias_cols(int K) { return (CODES16_TERMS * (K / 64) + 63) / 64 * 64; }
size_t codes16_bytes(int N, int K) { return (size_t)N * ((size_t)K * 2 + (size_t)codes16_bias_cols(K) * 2 + (size_t)(K / 64) * 4); }

// (float32 rows, whose biases are last, are multiplied by bf16 models' codes alone)
size_t codes16_kept_bytes(const LinearW& W) { return codes16_bytes(W.N, W.K) + (wk_scale_dtype(W.wk) == WK_BF16 ? (size_t)W.N * codes16_bias_cols(W.K) * 2 : 0); }

// side_only: biases and scales without the codes
static int codes16_into(const LinearW& src, void* codes, uint16_t* wb, float* sc, hipStream_t st, bool big_first, bool side_only) {
  const int bits = wk_bits(src.wk), sdt = wk_scale_dtype(src.wk);
  if (src.layout != 1 || (bits != 4 && bits != 8) || sdt == WK_F32 || src.group != 64 || src.K % (bits == 4 ? 128 : 64) != 0 || src.N % 16 != 0)
    return fail(MI_ERR_UNSUPPORTED, "codes16: tile-major int4 / int8 (group 64) matrices only");
  const int kb = codes16_bias_cols(src.K);
  const int nb = src.K / (bits == 4 ? 128 : 64), tiles = src.N / 16;
  const dim3 grid(side_only ? 1 : 1 + (nb + 7) / 8, tiles);          // (two blocks a wave)
#define GO(T, B) hipLaunchKernelGGL((codes16_kernel<T, B>), grid, dim3(256), (size_t)(src.K / 64) * 64, st, (const uint8_t*)src.w, (T*)codes, wb, sc, src.K, kb, (int)big_first)
  if (sdt == WK_BF16) { if (bits == 4) GO(bf16, 4); else GO(bf16, 8); }
  else { if (bits == 4) GO(f16, 4); else GO(f16, 8); }
#undef GO
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_codes16(const LinearW& src, void* dst, hipStream_t st, bool big_first) {
  char* d = (char*)dst;
  return codes16_into(src, d, (uint16_t*)(d + (size_t)src.N * src.K * 2), (float*)(d + (size_t)src.N * (src.K + codes16_bias_cols(src.K)) * 2), st, big_first, false);
}

int launch_codes16_kept(const LinearW& src, void* dst, hipStream_t st, Codes16& out) {
  char* d = (char*)dst;
  const bool both = wk_scale_dtype(src.wk) == WK_BF16;
  uint16_t* wb[2] = {(uint16_t*)(d + (size_t)src.N * src.K * 2), both ? (uint16_t*)(d + codes16_bytes(src.N, src.K)) : nullptr};
  float* sc = (float*)(d + (size_t)src.N * (src.K + codes16_bias_cols(src.K)) * 2);
  for (int f32 = 0; f32 < 1 + both; ++f32) MI_TRY(codes16_into(src, d, wb[f32], sc, st, f32 == 0, f32 == 1));
  out.codes = d; out.bias[0] = wb[0]; out.bias[1] = wb[1]; out.scales = sc;
  return MI_OK;
}

Codes16 codes16_rows(const Codes16& c, int n0, int K) {
  Codes16 r = c;
  if (c.codes == nullptr) return r;
  r.codes = (const char*)c.codes + (size_t)n0 * K * 2;
  for (int f32 = 0; f32 < 2; ++f32) r.bias[f32] = c.bias[f32] != nullptr ? (const char*)c.bias[f32] + (size_t)n0 * codes16_bias_cols(K) * 2 : nullptr;
  r.scales = c.scales + (size_t)n0 * (K / 64);
  return r;
}

size_t dequant_hilo_bytes(int N, int K) { return (size_t)N * K * 2 * 2; }

int launch_dequant_q4_hilo(const LinearW& src, void* dst, hipStream_t st) {
  const bool q4 = src.wk == WK_Q4_BF16 || src.wk == WK_Q4_F16, q8 = src.wk == WK_Q8_BF16 || src.wk == WK_Q8_F16;
  if (src.layout != 1 || (!q4 && !q8) || src.group != 64 || src.K % (q4 ? 128 : 64) != 0 || src.N % 16 != 0)
    return fail(MI_ERR_UNSUPPORTED, "dequant: tile-major int4 / int8 (group 64) matrices only");
  const dim3 grid(4096), block(256);
  if (src.wk == WK_Q4_BF16) hipLaunchKernelGGL(dequant_q4_hilo_kernel<bf16>, grid, block, 0, st, (const uint8_t*)src.w, (bf16*)dst, src.N, src.K);
  else if (src.wk == WK_Q4_F16) hipLaunchKernelGGL(dequant_q4_hilo_kernel<f16>, grid, block, 0, st, (const uint8_t*)src.w, (f16*)dst, src.N, src.K);
  else if (src.wk == WK_Q8_BF16) hipLaunchKernelGGL(dequant_q8_hilo_kernel<bf16>, grid, block, 0, st, (const uint8_t*)src.w, (bf16*)dst, src.N, src.K);
  else hipLaunchKernelGGL(dequant_q8_hilo_kernel<f16>, grid, block, 0, st, (const uint8_t*)src.w, (f16*)dst, src.N, src.K);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

bool tiled_supported(int wk, int N, int K, int group) {
  if (N % 16 != 0) return false;
  if (wk == WK_BF16 || wk == WK_F16) return K % 32 == 0;
  if (wk == WK_Q4_BF16 || wk == WK_Q4_F16) return group == 64 && K % 128 == 0;
  if (wk == WK_Q8_BF16 || wk == WK_Q8_F16) return group == 64 && K % 64 == 0;
  return false;
}

size_t tiled_bytes(int wk, int N, int K) {
  if (wk == WK_BF16 || wk == WK_F16) return (size_t)N * K * 2;
  if (wk == WK_Q8_BF16 || wk == WK_Q8_F16) return (size_t)(N / 16) * (K / 64) * 1088;
  // (+ 64 KiB: room behind the last tile for a stream that prefetches past its slice's end; what it loads there is never multiplied)
  return (size_t)(N / 16) * (K / 128) * 1152 + ((size_t)64 << 10);
}

int launch_repack_tiled(const LinearW& src, void* dst, hipStream_t st) {
  if (!tiled_supported(src.wk, src.N, src.K, src.group)) return fail(MI_ERR_UNSUPPORTED, "repack: matrix not eligible for the tile-major layout");
  if (src.layout != 0) return fail(MI_ERR_INVALID, "repack: source is not row-major");
  const dim3 grid(2048), block(256);
  if (src.wk == WK_BF16 || src.wk == WK_F16)
    hipLaunchKernelGGL(repack_dense16_kernel, grid, block, 0, st, (const uint16_t*)src.w, (uint16_t*)dst, src.N, src.K);
  else if (src.wk == WK_Q8_BF16 || src.wk == WK_Q8_F16)
    hipLaunchKernelGGL(repack_q8_kernel, grid, block, 0, st, (const uint32_t*)src.w, (const uint16_t*)src.scales,
                       (const uint16_t*)src.biases, (uint8_t*)dst, src.N, src.K);
  else
    hipLaunchKernelGGL(repack_q4_kernel, grid, block, 0, st, (const uint32_t*)src.w, (const uint16_t*)src.scales,
                       (const uint16_t*)src.biases, (uint8_t*)dst, src.N, src.K);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// Tile-major f16 matrix (N x K) -> tile-major bf16 matrix (N x 2K) whose columns [0, K) hold hi = bf16(w) and [K, 2K) hold
// lo = bf16(w - hi).  An f16 value has 11 significant bits and the bf16 range covers f16's, so hi + lo == w EXACTLY: the
// float32-activation kernels (x split exactly into three bf16 terms) then compute x . w as a float32 dot product of exact
// products for an f16 model too (PagedKVCache mode of the reference: base.py:111-112 promotes everything behind layer 0 to
// float32 whatever the model dtype).  The conversion keeps a block's lane order: block (tile t, k block j) of w becomes
// blocks (t, j) and (t, K / 32 + j) of the result.
__global__ void f16_to_hilo_kernel(const uint16_t* src, uint16_t* dst, int N, int K) {
  const size_t pieces = (size_t)N * (K / 8);
  const size_t kb = (size_t)(K / 32);
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < pieces; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t blk = idx >> 6, lane = idx & 63;
    const size_t t = blk / kb, j = blk % kb;
    const u32x4 v = *(const u32x4*)(src + idx * 8);
    const _Float16* h = (const _Float16*)&v;
    __bf16 hi[8], lo[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float w = (float)h[i];
      hi[i] = (__bf16)w;
      lo[i] = (__bf16)(w - (float)hi[i]);
    }
    *(u32x4*)(dst + ((t * 2 * kb + j) * 64 + lane) * 8) = *(const u32x4*)hi;
    *(u32x4*)(dst + ((t * 2 * kb + kb + j) * 64 + lane) * 8) = *(const u32x4*)lo;
  }
}

// Row-interleaved copy of a tile-major gate|up matrix for the decode GEMV (gemv_mfma, EPI_SWIGLU_GU8).  With gate and up
// as separate 16-row tiles a SwiGLU work item is a PAIR of tiles, and 14336 / 16 = 896 pairs deal 3.5 to each of 256 CUs:
// half the CUs stream a fourth pair while the others idle (12.5 % of the launch).  Tile t of the copy holds gate rows
// 8t .. 8t+7 in its rows 0..7 and up rows 8t .. 8t+7 in rows 8..15: 1792 one-tile items, 7 per CU, same bytes per item as
// any plain tile, and silu(g) * u pairs columns j and j + 8 of one MFMA tile.  16-byte pieces: lane (g, c16) of block
// (tile, k block) holds 8 k of row c16.
__global__ __launch_bounds__(256) void gate_up_interleave_kernel(const u32x4* src, u32x4* dst, int I, int kblocks, size_t total) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int l = (int)(i & 63), c16 = l & 15, g = l >> 4;
  const size_t blk = i >> 6;
  const int kb = (int)(blk % kblocks);
  const int t = (int)(blk / kblocks);
  const int row = c16 < 8 ? 8 * t + c16 : I + 8 * t + (c16 - 8);
  dst[i] = src[((size_t)(row >> 4) * kblocks + kb) * 64 + g * 16 + (row & 15)];
}

int launch_gate_up_interleave(const LinearW& W, int pair_offset, void* dst, hipStream_t st) {
  if (W.layout != 1 || (W.wk != WK_BF16 && W.wk != WK_F16) || W.N != 2 * pair_offset || pair_offset % 16 != 0 || W.K % 32 != 0)
    return fail(MI_ERR_INVALID, "gate_up_interleave: a tile-major dense 16-bit gate|up matrix with pair_offset % 16 == 0");
  const size_t total = (size_t)W.N * W.K * 2 / 16;
  hipLaunchKernelGGL(gate_up_interleave_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, (const u32x4*)W.w, (u32x4*)dst,
                     pair_offset, W.K / 32, total);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_f16_to_hilo(const LinearW& tiled_f16, void* dst, hipStream_t st) {
  if (tiled_f16.wk != WK_F16 || tiled_f16.layout != 1) return fail(MI_ERR_INVALID, "f16_to_hilo: a tile-major f16 matrix is expected");
  hipLaunchKernelGGL(f16_to_hilo_kernel, dim3(2048), dim3(256), 0, st, (const uint16_t*)tiled_f16.w, (uint16_t*)dst, tiled_f16.N, tiled_f16.K);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
