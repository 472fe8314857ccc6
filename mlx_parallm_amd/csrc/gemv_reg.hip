// gemv_reg.hip -- decode linears of at most 8 rows, activations in registers: int4 / int8 weights, and (gemv_dense_kernel) 16-bit ones: y[M][N] = x[M][K] . W[N][K]^T
// (nn.QuantizedLinear call sites llama.py:64-67,93,143,160-165,250-252; qwen3.py:37-40,63,115).
//
// The split-K kernel of gemm_skinny.hip spends most of a short launch outside the weight stream: x goes through LDS in chunks with a
// barrier each, the K slices of a tile meet through memory (write-through stores, a counter, a read-back: 3 us of an 11-us launch),
// and the norm in front needs the producer's partial sums.  Here a workgroup of 8 waves owns whole output tiles of 16 columns, its
// waves split K, and a wave keeps ITS columns of x -- 8 rows x at most 640 -- as MFMA A-fragments in registers: 16-byte loads straight
// from the row-major x, no LDS image, no barrier in front of the first product.  All waves together hold whole rows, so the RMS norm
// costs one exchange of sums through LDS, under the flight of the first weight blocks.  The waves' partial tiles meet in LDS (one
// barrier per tile, two buffers); nothing crosses workgroups.  Tiles are dealt round-robin to one workgroup per CU, and the weight
// loads of the next tile go out as the registers of this one are consumed (none behind the last: a pass of 8 rows 10.4 -> 10.1 ms).
//
// gemv_long_kernel: K beyond that (int4 down_proj), no norm.  One tile per workgroup, every block's x fragments loaded next to it
// (from L2), 12 blocks in flight per wave.
//
// Quantised weights: per 64-group y += s sum(q x) + (b - offs s) sum(x); sum(x) of a group is an MFMA of the same fragments with ones,
// whose result already lies in the accumulator's layout.
//
// Measured (Mistral-7B shapes, 8 rows, rocprof us, gemm_skinny.hip -> here; an empty kernel is 4): int4 q|k|v 11.3 -> 9.0, o 11.3 -> 6.4,
// gate|up 21.3 -> 17.7, down 15.0 -> 14.8; int8 (3 rows) o 11.6 -> 7.4.  The stream itself is 9 to 66 MB = 1.6 to 11.2 us (int4); what is
// left is the norm in front (2.5 us) and, in down, ~75 vector instructions per block.  The error against 64 bits is no larger than
// gemm_skinny.hip's: bf16 results that round to another value than the exact one 3.4e-4 / 3.4e-4 (int4, K 4096 / 14336; 3.4e-4 /
// 4.3e-4 there), int8 3e-5 (6e-5); dense 16-bit rows (K 1024 to 5120, with and without the norm; gemv_mfma.hip there) bf16 1.1e-4 (1.3e-4), f16
// 1.8e-3 (2.4e-3).
#include <algorithm>

#include "gemv_phase.h"

namespace mi {

int gemv_cu_count();      // gemv_mfma.hip

namespace {

using namespace gemv;

struct RegParams {
  const void* x; int ldx; int M;
  int norm; const void* norm_w; float eps;
  const void* w; int N, K;
  int epi; void* out; int ldo; void* resid; int pair_offset;
  int ntiles, nblk;              // 16-column tiles (pairs for SwiGLU), blocks of a tile along K
};

template <int QB> struct Blk;                                                    // one tile-major block: k, bytes, A-fragments
template <> struct Blk<4> { static constexpr int K = 128, BYTES = 1152, F = 4; };
template <> struct Blk<8> { static constexpr int K = 64, BYTES = 1088, F = 2; };

// k offset within a block of the 8 values that lane group g supplies to product i of the block
template <int QB>
__device__ __forceinline__ int frag_k(int i, int g) {
  if constexpr (QB == 4) return (i >> 1) * 64 + ((((g & 1) << 2) | ((g >> 1) << 1)) + (i & 1)) * 8;      // (gemv_phase.h: frag_slot)
  return g * 16 + i * 8;
}
// the order in which unpack_q4 leaves 8 codes: 0 4 1 5 2 6 3 7
__device__ __forceinline__ u32x4 nibble_order(u32x4 v) {
  return u32x4{__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
               __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
}
template <typename AT>
__device__ __forceinline__ u32x4 ones16() {
  const uint32_t o = std::is_same<AT, bf16>::value ? 0x3F803F80u : 0x3C003C00u;
  return u32x4{o, o, o, o};
}
// codes - 128: as much below as above zero, so that neither the products' sum nor the bias term (b + 128 s, about zero) is large against
// the result; -128 .. 127 are exact in bf16 and f16
template <typename AT>
__device__ __forceinline__ u32x4 unpack_q8(uint32_t lo, uint32_t hi) {
  lo ^= 0x80808080u; hi ^= 0x80808080u;
  u32x4 r;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    r[j] = pack2<AT>(f32x2{(float)(int8_t)(lo >> (16 * j)), (float)(int8_t)(lo >> (16 * j + 8))});
    r[2 + j] = pack2<AT>(f32x2{(float)(int8_t)(hi >> (16 * j)), (float)(int8_t)(hi >> (16 * j + 8))});
  }
  return r;
}

template <int QB> struct WBlk { u32x4 v; uint32_t s, b; };

template <typename AT, int QB>
__device__ __forceinline__ void load_blk(WBlk<QB>& w, const char* blk, int lane, int c16) {
  w.v = __builtin_nontemporal_load((const u32x4*)(blk + lane * 16));
  if constexpr (QB == 4) { w.s = *(const uint32_t*)(blk + 1024 + c16 * 4); w.b = *(const uint32_t*)(blk + 1088 + c16 * 4); }
  if constexpr (QB == 8) { w.s = *(const uint16_t*)(blk + 1024 + c16 * 2); w.b = *(const uint16_t*)(blk + 1056 + c16 * 2); }
}

// acc += the block's products; xf: its A-fragments, sx: its groups' sums of x
template <typename AT, int QB>
__device__ __forceinline__ void mul_blk(f32x4& acc, const WBlk<QB>& w, const u32x4* xf, const f32x4* sx) {
  constexpr int NG = QB == 4 ? 2 : 1;
  u32x4 q[2 * NG];
  if constexpr (QB == 4) {
    auto r0 = __builtin_amdgcn_permlane32_swap(w.v.x, w.v.z, false, false);
    auto r1 = __builtin_amdgcn_permlane32_swap(w.v.y, w.v.w, false, false);
    q[0] = unpack_q4<AT>(r0[0]); q[1] = unpack_q4<AT>(r1[0]);
    q[2] = unpack_q4<AT>(r0[1]); q[3] = unpack_q4<AT>(r1[1]);
  } else {
    q[0] = unpack_q8<AT>(w.v.x, w.v.y); q[1] = unpack_q8<AT>(w.v.z, w.v.w);
  }
  f32x4 d[NG];
#pragma unroll
  for (int j = 0; j < NG; ++j) d[j] = mfma16<AT>(xf[2 * j], q[2 * j], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int j = 0; j < NG; ++j) d[j] = mfma16<AT>(xf[2 * j + 1], q[2 * j + 1], d[j]);
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    const float sc = (float)__builtin_bit_cast(AT, (unsigned short)(w.s >> (16 * j)));
    const float bb = (float)__builtin_bit_cast(AT, (unsigned short)(w.b >> (16 * j))) - (QB == 4 ? Magic<AT>::offs : -128.f) * sc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = fmaf(sc, d[j][r], fmaf(bb, sx[j][r], acc[r]));
  }
}

__device__ __forceinline__ float sum_waves(const float* q) {      // the eight waves' partial tiles at one place
  return ((q[0] + q[256]) + (q[512] + q[768])) + ((q[1024] + q[1280]) + (q[1536] + q[1792]));
}

// y[m][n] of one tile (gate and up for SwiGLU), m = tid / 16, n = tile's column tid % 16: the waves' partial tiles added pairwise
template <typename AT, int NW, bool SW>
__device__ __forceinline__ void finish_tile(const RegParams& p, const float* part, int tile, int tid, float hv) {
  const int m = tid >> 4, n = tile * 16 + (tid & 15), at = ((m >> 2) * 16 + (tid & 15)) * 4 + (m & 3);
  static_assert(NW == 8, "");
  const float y = sum_waves(part + at), u = SW ? sum_waves(part + NW * 256 + at) : 0.f;
  AT* out = (AT*)p.out;
  if constexpr (SW) out[(size_t)m * p.ldo + n] = silu16<AT>(y, u);
  else if (p.epi == EPI_STORE) out[(size_t)m * p.ldo + n] = (AT)y;
  else if (p.epi == EPI_STORE_F32) ((float*)p.out)[(size_t)m * p.ldo + n] = (float)(AT)y;
  else ((AT*)p.resid)[(size_t)m * p.ldo + n] = (AT)(hv + (float)(AT)y);
}

// The A-fragments of two consecutive products in one register: rows 8 .. 15 of a product are nobody's, so the lanes of columns 8 .. 15
// load the SECOND fragment of rows 0 .. 7 -- half the loads -- and the second product takes the register rotated by eight lanes
// (the first one's rows 8 .. 15 are then numbers that nobody reads).
template <typename AT, int QB>
__device__ __forceinline__ u32x4 load_pair(const AT* row, int k0, int pair, int c16, int g) {      // row: of column c16 % 8
  return *(const u32x4*)(row + k0 + frag_k<QB>(2 * pair + (c16 >> 3), g));
}
__device__ __forceinline__ u32x4 ror8(u32x4 v) {
  u32x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = __builtin_amdgcn_update_dpp(0u, v[j], 0x128, 0xf, 0xf, false);
  return r;
}

// KW: k per wave, at most; FULL: every wave has that.  Otherwise a wave with less loads its last block again, and skips it -- zero
// fragments would do for finite weights, but 0 x inf is NaN.  The skip's branches cost 0.1 to 0.5 us a launch (o of Mistral-7B in bf16 7.9 -> 8.4),
// so the full shares have none.
template <typename AT, int QB, bool SW, bool NORM, int KW, bool FULL>
__global__ __launch_bounds__(512, 2) void gemv_reg_kernel(const RegParams p) {
  using B = Blk<QB>;
  constexpr int NW = 8, NA = SW ? 2 : 1, NB = KW / B::K, NP = KW / 64, PB = B::F / 2;     // pairs of fragments: in all, per block
  __shared__ __attribute__((aligned(16))) float part[2][NA * NW * 256];
  __shared__ float sq[NW][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
  const int b0 = wave * p.nblk / NW, nb = (wave + 1) * p.nblk / NW - b0;        // this wave's blocks of every tile

  WBlk<QB> wb[NA][NB];
  const size_t tile_bytes = (size_t)p.nblk * B::BYTES;
  const int step = gridDim.x;
  auto issue = [&](int a, int i, int tile) {
    const char* t = (const char*)p.w + (size_t)(tile + a * (p.pair_offset >> 4)) * tile_bytes;
    load_blk<AT, QB>(wb[a][i], t + (size_t)(b0 + min(i, max(nb - 1, 0))) * B::BYTES, lane, c16);
  };
  auto issue_first = [&] {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int a = 0; a < NA; ++a) issue(a, i, blockIdx.x);
  };
  // A wave's loads return in order.  Without a norm the first tile's blocks go out first, x from L2 arrives right behind them; with one, x
  // and the norm's weights are in front and the norm runs under the blocks' flight (int4 gate|up 19.1 against 17.7 us, q|k|v 9.4 / 9.0).
  if constexpr (!NORM) issue_first();

  // ---- x: rows beyond M are clamped (their products are nobody's)
  u32x4 xf[NP];
  const AT* xr = (const AT*)p.x + (size_t)min(c16 & 7, p.M - 1) * p.ldx;
  auto k_of = [&](int q) { return (b0 + min(q / PB, max(nb - 1, 0))) * B::K; };
#pragma unroll
  for (int q = 0; q < NP; ++q) xf[q] = load_pair<AT, QB>(xr, k_of(q), q % PB, c16, g);
  u32x4 nw[NORM ? NP : 1];
  if constexpr (NORM) {
#pragma unroll
    for (int q = 0; q < NP; ++q) nw[q] = load_pair<AT, QB>((const AT*)p.norm_w, k_of(q), q % PB, c16, g);
    __builtin_amdgcn_sched_barrier(0);
    issue_first();
  }
  // residual: nobody else writes these columns
  const bool res = !SW && p.epi == EPI_RESID, fin = tid < 256 && (tid >> 4) < p.M;
  const AT* hrow = (const AT*)(res ? p.resid : p.x) + (res ? (size_t)min(tid >> 4, p.M - 1) * p.ldo + (tid & 15) : 0);
  __builtin_amdgcn_sched_barrier(0);

  if constexpr (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      float s1 = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) { const f32x2 e = unpack2<AT>(xf[q][j]); s1 = fmaf(e.x, e.x, fmaf(e.y, e.y, s1)); }
      ss += q / PB < nb ? s1 : 0.f;
    }
    ss += __builtin_amdgcn_update_dpp(0.f, ss, 0x128, 0xf, 0xf, false);      // (columns c and c + 8 hold one row)
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) sq[wave][c16] = ss;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) t += sq[w][c16];
    const float rs = 1.0f / sqrtf(t / (float)p.K + p.eps);
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {                   // w * cast_T(x32 * rsqrt(..)), rounded to T
        const f32x2 e = unpack2<AT>(xf[q][j]), we = unpack2<AT>(nw[q][j]);
        const f32x2 xn = unpack2<AT>(pack2<AT>(f32x2{e.x * rs, e.y * rs}));
        xf[q][j] = pack2<AT>(f32x2{xn.x * we.x, xn.y * we.y});
      }
  }
  f32x4 sx[NP];
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    if constexpr (QB == 4) xf[q] = nibble_order(xf[q]);
    sx[q] = mfma16<AT>(xf[q], ones16<AT>(), f32x4{0.f, 0.f, 0.f, 0.f});
    sx[q] = mfma16<AT>(ror8(xf[q]), ones16<AT>(), sx[q]);
  }

  int buf = 0;
  auto do_tile = [&](int tile, auto more) {           // (more: another tile follows)
    const AT hv = hrow[res ? tile * 16 : 0];
    f32x4 acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      u32x4 f[B::F];
#pragma unroll
      for (int q = 0; q < PB; ++q) { f[2 * q] = xf[i * PB + q]; f[2 * q + 1] = ror8(xf[i * PB + q]); }
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        if (FULL || i < nb) mul_blk<AT, QB>(acc[a], wb[a][i], f, sx + i * PB);      // (uniform)
        if constexpr (decltype(more)::value) {
          __builtin_amdgcn_sched_barrier(0);
          issue(a, i, tile + step);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) *(f32x4*)&part[buf][(a * NW + wave) * 256 + lane * 4] = acc[a];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                     // (the loads of the next tile stay in flight)
    asm volatile("" ::: "memory");
    if (fin) finish_tile<AT, NW, SW>(p, part[buf], tile, tid, (float)hv);
    buf ^= 1;                                         // the buffer read now is written again two tiles on, behind the next barrier
  };
  int tile = blockIdx.x;
  for (; tile + step < p.ntiles; tile += step) do_tile(tile, std::true_type{});
  do_tile(tile, std::false_type{});
}

// NB: int4 blocks per wave, at most
template <typename AT, int NB>
__global__ __launch_bounds__(512, 2) void gemv_long_kernel(const RegParams p) {
  constexpr int QB = 4;
  using B = Blk<QB>;
  constexpr int NW = 8, PB = B::F / 2, R = NB < 12 ? NB : 12;      // blocks in flight per wave: what 256 registers hold
  __shared__ __attribute__((aligned(16))) float part[NW * 256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
  const int b0 = wave * p.nblk / NW, nb = (wave + 1) * p.nblk / NW - b0, tile = blockIdx.x;
  const AT* xr = (const AT*)p.x + (size_t)min(c16 & 7, p.M - 1) * p.ldx;
  const char* wt = (const char*)p.w + (size_t)tile * p.nblk * B::BYTES;
  u32x4 xf[R][PB];
  WBlk<QB> wb[R];
  auto issue = [&](int i) {                           // (past the last block: the last one again, unused)
    const int b = b0 + min(i, max(nb - 1, 0));
    load_blk<AT, QB>(wb[i % R], wt + (size_t)b * B::BYTES, lane, c16);
#pragma unroll
    for (int q = 0; q < PB; ++q) xf[i % R][q] = load_pair<AT, QB>(xr, b * B::K, q, c16, g);
  };
#pragma unroll
  for (int i = 0; i < R; ++i) issue(i);
  const bool res = p.epi == EPI_RESID, fin = tid < 256 && (tid >> 4) < p.M;
  const AT hv = ((const AT*)(res ? p.resid : p.x))[res ? (size_t)min(tid >> 4, p.M - 1) * p.ldo + tile * 16 + (tid & 15) : 0];
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (i < nb) {                                     // (uniform)
      u32x4 f[B::F];
      f32x4 sx[PB];
#pragma unroll
      for (int q = 0; q < PB; ++q) {
        f[2 * q] = nibble_order(xf[i % R][q]);
        f[2 * q + 1] = ror8(f[2 * q]);
        sx[q] = mfma16<AT>(f[2 * q], ones16<AT>(), f32x4{0.f, 0.f, 0.f, 0.f});
        sx[q] = mfma16<AT>(f[2 * q + 1], ones16<AT>(), sx[q]);
      }
      mul_blk<AT, QB>(acc, wb[i % R], f, sx);
    }
    if (i + R < NB) {
      __builtin_amdgcn_sched_barrier(0);
      issue(i + R);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  *(f32x4*)&part[wave * 256 + lane * 4] = acc;
  __syncthreads();
  if (fin) finish_tile<AT, NW, false>(p, part, tile, tid, (float)hv);
}

// Dense 16-bit weights, x in float32 (the float32-cache mode; X32) or in the weights' type.  The same split of the work; x is split exactly
// into three terms of the weights' type in registers (96 of them at 512 k per wave), each weight fragment meets the three, their sums stay
// apart up to the end.  A tile's 16 fragments are all in flight, the next tile's go out as they are consumed.
// GU: tiles of the row-interleaved gate|up copy (8 gate, 8 up rows; repack.hip): seven per CU where whole pairs are 3.5.
// Measured (Mistral-7B shapes, rocprof us; an empty kernel is 4).  float32 x, 8 rows, gemm_skinny.hip -> here: gate|up 50.6 -> 43.0 (235 MB at
// the card's 5.9 TB/s: 41.7; 224 workgroups there), q|k|v 17.0 -> 15.7, o 13.1 -> 11.3; its rms error against 64 bits is 0.4 of that kernel's.
// 16-bit x, 1 row, gemv_mfma.hip -> here: q|k|v and o 12.6 on average -> 11.0 and 7.9; K = 2048, 4 rows 18.3 -> 10.3.
template <typename AT, bool X32>
struct RawX { u32x4 v[X32 ? 2 : 1]; };
template <typename AT, bool X32>
__device__ __forceinline__ void unpack_raw(const RawX<AT, X32>& r, f32x2 (&e)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (X32) e[j] = f32x2{__uint_as_float(r.v[j >> 1][2 * (j & 1)]), __uint_as_float(r.v[j >> 1][2 * (j & 1) + 1])};
    else e[j] = unpack2<AT>(r.v[0][j]);
  }
}

template <typename AT, bool X32, bool GU, bool NORM, int KW, bool FULL>       // (KW, FULL: as gemv_reg_kernel)
__global__ __launch_bounds__(512, 2) void gemv_dense_kernel(const RegParams p) {
  using XT = typename std::conditional<X32, float, AT>::type;
  constexpr int NW = 8, NP = KW / 32, NQ = NP / 2, T = X32 ? 3 : 1, NC = X32 ? 3 : 2;      // products, pairs of them, terms, chains of sums
  __shared__ __attribute__((aligned(16))) float part[2][NW * 256];
  __shared__ float sq[NW][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
  const int q0 = wave * p.nblk / NW, nq = (wave + 1) * p.nblk / NW - q0;        // this wave's pairs (64 k each) of every tile
  const int step = gridDim.x;

  u32x4 wb[NP];
  auto pair_at = [&](int q) { return q0 + min(q, max(nq - 1, 0)); };            // (past the last: the last one again, unused)
  auto issue = [&](int i, int tile) {
    wb[i] = __builtin_nontemporal_load((const u32x4*)((const char*)p.w + ((size_t)tile * p.nblk * 2 + pair_at(i >> 1) * 2 + (i & 1)) * 1024 + lane * 16));
  };
  auto issue_first = [&] {
#pragma unroll
    for (int i = 0; i < NP; ++i) issue(i, blockIdx.x);
  };
  if constexpr (!NORM) issue_first();

  RawX<AT, X32> raw[NQ], nw[NORM ? NQ : 1];
  const int koff = (c16 >> 3) * 32 + g * 8;                                     // lanes of columns 8 .. 15: the pair's second fragment
  const XT* xr = (const XT*)p.x + (size_t)min(c16 & 7, p.M - 1) * p.ldx + koff;
  auto load_raw = [&](RawX<AT, X32>& r, const XT* s, int q) {
#pragma unroll
    for (int h = 0; h < (X32 ? 2 : 1); ++h) r.v[h] = *(const u32x4*)(s + pair_at(q) * 64 + h * 4);
  };
#pragma unroll
  for (int q = 0; q < NQ; ++q) load_raw(raw[q], xr, q);
  if constexpr (NORM) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) load_raw(nw[q], (const XT*)p.norm_w + koff, q);
    __builtin_amdgcn_sched_barrier(0);
    issue_first();
  }
  __builtin_amdgcn_sched_barrier(0);
  const bool res = !GU && p.epi == EPI_RESID, fin = tid < 256 && (tid >> 4) < p.M;
  const XT* hrow = (const XT*)(res ? p.resid : p.x) + (res ? (size_t)min(tid >> 4, p.M - 1) * p.ldo + (tid & 15) : 0);

  float rs = 1.f;
  if constexpr (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      f32x2 e[4];
      unpack_raw<AT, X32>(raw[q], e);
      float s1 = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) s1 = fmaf(e[j].x, e[j].x, fmaf(e[j].y, e[j].y, s1));
      ss += q < nq ? s1 : 0.f;
    }
    ss += __builtin_amdgcn_update_dpp(0.f, ss, 0x128, 0xf, 0xf, false);      // (columns c and c + 8 hold one row)
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) sq[wave][c16] = ss;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) t += sq[w][c16];
    rs = 1.0f / sqrtf(t / (float)p.K + p.eps);
  }
  u32x4 xf[T][NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    f32x2 e[4], we[4];
    unpack_raw<AT, X32>(raw[q], e);
    if constexpr (NORM) unpack_raw<AT, X32>(nw[q], we);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (X32) {
        f32x2 v = e[j];
        if constexpr (NORM) v = f32x2{v.x * rs * we[j].x, v.y * rs * we[j].y};
        const uint32_t hi = pack2<AT>(v);
        const f32x2 h = unpack2<AT>(hi), r1 = f32x2{v.x - h.x, v.y - h.y};
        const uint32_t mid = pack2<AT>(r1);
        const f32x2 m = unpack2<AT>(mid);
        xf[0][q][j] = hi; xf[1][q][j] = mid; xf[2][q][j] = pack2<AT>(f32x2{r1.x - m.x, r1.y - m.y});
      } else if constexpr (NORM) {                    // w * cast_T(x32 * rsqrt(..)), rounded to T
        const f32x2 xn = unpack2<AT>(pack2<AT>(f32x2{e[j].x * rs, e[j].y * rs}));
        xf[0][q][j] = pack2<AT>(f32x2{xn.x * we[j].x, xn.y * we[j].y});
      } else {
        xf[0][q][j] = raw[q].v[0][j];
      }
    }
  }

  int buf = 0;
  auto do_tile = [&](int tile, auto more) {
    const XT hv = hrow[res ? tile * 16 : 0];
    f32x4 acc[NC];
#pragma unroll
    for (int a = 0; a < NC; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (FULL || i < 2 * nq) {                       // (uniform)
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const u32x4 f = (i & 1) ? ror8(xf[t][i >> 1]) : xf[t][i >> 1];
          f32x4& a = acc[X32 ? t : i & 1];
          a = mfma16<AT>(f, wb[i], a);
        }
      }
      if constexpr (decltype(more)::value) {
        __builtin_amdgcn_sched_barrier(0);
        issue(i, tile + step);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    *(f32x4*)&part[buf][wave * 256 + lane * 4] = X32 ? (acc[NC - 1] + acc[1]) + acc[0] : acc[0] + acc[1];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                     // (the loads of the next tile stay in flight)
    asm volatile("" ::: "memory");
    if constexpr (!X32) {
      if (fin) finish_tile<AT, NW, false>(p, part[buf], tile, tid, (float)hv);
    } else if (fin) {
      const int m = tid >> 4, c = tid & 15, at = ((m >> 2) * 16 + c) * 4 + (m & 3);
      const float y = sum_waves(part[buf] + at);
      if constexpr (GU) {
        const float u = __shfl_down(y, 8);
        if (c < 8) {
          const float sig = 1.0f / (1.0f + expf(-y)), sl = y * sig;
          ((float*)p.out)[(size_t)m * p.ldo + tile * 8 + c] = sl * u;
        }
      } else if (res) ((float*)p.resid)[(size_t)m * p.ldo + tile * 16 + c] = hv + y;
      else ((float*)p.out)[(size_t)m * p.ldo + tile * 16 + c] = y;
    }
    buf ^= 1;                                         // the buffer read now is written again two tiles on, behind the next barrier
  };
  int tile = blockIdx.x;
  for (; tile + step < p.ntiles; tile += step) do_tile(tile, std::true_type{});
  do_tile(tile, std::false_type{});
}

// The output linear of a layer with a token input (layer_rows.hip: side_join_kernel reads what this leaves), 16-bit weights and rows.  A tile and a slice of K per workgroup,
// so that a width of 2048 (128 tiles) fills the card: part[s][m][n] = the slice's sums, with the residual in slice 0; and of those 16 columns each gate output's share,
// z[s tiles + tile][m][j] = sum_n gate[j][n] part[s][m][n], so that no workgroup of what follows reads the gate's matrix.
// 4 rows, 2048 x 10240 bf16, us in a decode step: gemv_mfma.hip 15.6 and the gate, projection and norms of a row in one workgroup 12.2; here 10.3 and 9.3 (a layer 53 -> 46).
struct SideParams {
  const void* x; int ldx; int M;
  const void* w; int nblk, ks;
  const float* resid; int ld;
  const void* gate; int dim;
  float* part; float* z;
};
template <typename AT, int KW, bool FULL>             // (KW, FULL: as gemv_reg_kernel, of a slice)
__global__ __launch_bounds__(512, 2) void gemv_side_kernel(const SideParams p) {
  constexpr int NW = 8, NP = KW / 32, NQ = NP / 2;
  __shared__ __attribute__((aligned(16))) float tl[NW * 256];
  __shared__ __attribute__((aligned(16))) float xs[8][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
  const int tile = blockIdx.x, s = blockIdx.y, sn = p.nblk / p.ks;                     // (slices of whole pairs: the host)
  const int q0 = s * sn + wave * sn / NW, nq = (wave + 1) * sn / NW - wave * sn / NW;
  auto pair_at = [&](int q) { return q0 + min(q, max(nq - 1, 0)); };                   // (past the last: the last one again, unused)
  u32x4 wb[NP], xf[NQ], gw[2];
#pragma unroll
  for (int i = 0; i < NP; ++i)
    wb[i] = __builtin_nontemporal_load((const u32x4*)((const char*)p.w + ((size_t)tile * p.nblk * 2 + pair_at(i >> 1) * 2 + (i & 1)) * 1024 + lane * 16));
  const AT* xr = (const AT*)p.x + (size_t)min(c16 & 7, p.M - 1) * p.ldx + (c16 >> 3) * 32 + g * 8;
#pragma unroll
  for (int q = 0; q < NQ; ++q) xf[q] = *(const u32x4*)(xr + pair_at(q) * 64);
  const AT* gr = (const AT*)p.gate + (size_t)min(lane, p.dim - 1) * p.ld + tile * 16;
#pragma unroll
  for (int h = 0; h < 2; ++h) gw[h] = *(const u32x4*)(gr + 8 * h);
  const int m = min(tid >> 4, p.M - 1), n = tile * 16 + (tid & 15);
  const float r0 = p.resid[(size_t)m * p.ld + n];
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (FULL || i < 2 * nq) acc[i & 1] = mfma16<AT>((i & 1) ? ror8(xf[i >> 1]) : xf[i >> 1], wb[i], acc[i & 1]);      // (uniform)
  *(f32x4*)&tl[wave * 256 + lane * 4] = acc[0] + acc[1];
  __syncthreads();
  if (tid < 128) {
    const float y = sum_waves(tl + (((tid >> 6) * 16 + (tid & 15)) * 4 + ((tid >> 4) & 3))) + (s == 0 ? r0 : 0.f);
    xs[tid >> 4][tid & 15] = y;
    if ((tid >> 4) < p.M) p.part[((size_t)s * p.M + (tid >> 4)) * p.ld + n] = y;
  }
  __syncthreads();
  if (wave < p.M && lane < p.dim) {                   // row `wave`, gate output `lane`
    float z = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x2 e = unpack2<AT>(gw[h][j]);
        z = fmaf(e.x, xs[wave][8 * h + 2 * j], fmaf(e.y, xs[wave][8 * h + 2 * j + 1], z));
      }
    p.z[(((size_t)s * gridDim.x + tile) * p.M + wave) * 64 + lane] = z;
  }
}

int quant_bits(const LinearW& W, int act) {           // 4 / 8: codes with scales of the activation type, 0: neither
  if (((W.wk == WK_Q4_BF16 && act == MI_BF16) || (W.wk == WK_Q4_F16 && act == MI_F16)) && W.group == 64) return 4;
  if (((W.wk == WK_Q8_BF16 && act == MI_BF16) || (W.wk == WK_Q8_F16 && act == MI_F16)) && W.group == 64) return 8;
  return 0;
}
// Longest K whose activations stay in registers; longest K at all.  The second is no limit of the kernel (its registers do not grow past 12
// blocks a wave): it is the longest that was measured, and what is longer stays on gemm_skinny.hip.
constexpr int REG_K = 8 * 640, LONG_K = 8 * 17 * 128;

}  // namespace

bool gemv_reg_supported(const LinearW& W, const GemvCall& c, size_t rows) {
  static const bool off = getenv("MI_GEMV_REG") != nullptr && atoi(getenv("MI_GEMV_REG")) == 0;      // (A/B)
  if (off || c.force_v1 || W.layout != 1 || rows < 1 || rows > 8 || c.act == MI_F32 || c.rnd != RND_NONE) return false;
  if (W.lora_b[0] != nullptr || W.lora_b[1] != nullptr || c.out32 || c.silu_cols > 0 || c.glu.kind != GLU_SILU) return false;
  if (c.epi != EPI_STORE && c.epi != EPI_STORE_F32 && c.epi != EPI_RESID && c.epi != EPI_SWIGLU) return false;
  const int qb = quant_bits(W, c.act), bk = qb == 4 ? 128 : 64, n = c.epi == EPI_SWIGLU ? c.pair_offset : W.N;
  if (qb == 0 || W.K % bk != 0 || n % 16 != 0 || W.K > LONG_K) return false;
  if (W.K > REG_K && (c.pro == PRO_NORM || c.epi == EPI_SWIGLU)) return false;
  if (c.epi == EPI_SWIGLU && c.pro != PRO_NORM) return false;      // (no caller)
  // int8: o_proj and the head (11.6 -> 7.4 and 29.6 -> 26 us).  The other three would gain 1.4 to 2.4 us each (q|k|v 13.5 -> 11.5, gate|up
  // 26.6 -> 25.2, down 17.4 -> 15.0), but any other order of their sums than gemm_skinny.hip's lets one of the recorded greedy sequences
  // fall to the fourth of five candidates one ulp of a bf16 logit apart, and those sequences stay as they are.
  if (qb == 8 && (W.K > REG_K || c.epi == EPI_SWIGLU || (c.pro == PRO_NORM && c.epi != EPI_STORE_F32))) return false;
  // 16-byte loads of x and the norm's weights
  return c.ldx % 8 == 0 && (uintptr_t)c.x % 16 == 0 && (c.pro != PRO_NORM || (uintptr_t)c.norm_w % 16 == 0);
}

// f(k per wave of the instantiation, every wave has that): the smallest registers that hold a wave's blocks of bk.
// FULL640 = false: the largest never takes the branchless form (with three terms of x and the norm that one spills three registers)
template <bool FULL640 = true, class F>
static int by_share(int nblk, int bk, F f) {
  auto at = [&](auto kw) {
    if constexpr (FULL640 || kw.value < 640)
      if (nblk * bk == 8 * kw) return f(kw, std::true_type{});
    return f(kw, std::false_type{});
  };
  const int kw = (nblk + 7) / 8 * bk;
  return kw <= 256 ? at(std::integral_constant<int, 256>{}) : kw <= 512 ? at(std::integral_constant<int, 512>{}) : at(std::integral_constant<int, 640>{});
}

template <typename AT, int QB>
static int launch_reg(const RegParams& p, bool sw, hipStream_t st) {
  auto go = [&](auto kern, int grid) -> int {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), 0, st, p);
    MI_HIP(hipGetLastError());
    return MI_OK;
  };
  const int grid = std::min(p.ntiles, gemv_cu_count());
  if constexpr (QB == 4) {
    if (p.K > REG_K) {
      const int nb = (p.nblk + 7) / 8;
      if (nb <= 8) return go(gemv_long_kernel<AT, 8>, p.ntiles);
      if (nb <= 11) return go(gemv_long_kernel<AT, 11>, p.ntiles);
      if (nb <= 14) return go(gemv_long_kernel<AT, 14>, p.ntiles);
      return go(gemv_long_kernel<AT, 17>, p.ntiles);
    }
    if (sw) return by_share(p.nblk, 128, [&](auto kw, auto full) { return go(gemv_reg_kernel<AT, 4, true, true, kw.value, full.value>, grid); });
  }
  if (p.norm) return by_share(p.nblk, Blk<QB>::K, [&](auto kw, auto full) { return go(gemv_reg_kernel<AT, QB, false, true, kw.value, full.value>, grid); });
  return by_share(p.nblk, Blk<QB>::K, [&](auto kw, auto full) { return go(gemv_reg_kernel<AT, QB, false, false, kw.value, full.value>, grid); });
}

int launch_gemv_reg(const LinearW& W, const GemvCall& c, size_t rows, hipStream_t st) {
  if (!gemv_reg_supported(W, c, rows)) return fail(MI_ERR_UNSUPPORTED, "gemv_reg: shape / dtype not supported");
  const int qb = quant_bits(W, c.act);
  const bool sw = c.epi == EPI_SWIGLU;
  RegParams p{};
  p.x = c.x; p.ldx = c.ldx; p.M = (int)rows;
  p.norm = c.pro == PRO_NORM; p.norm_w = c.norm_w; p.eps = c.eps;
  p.w = W.w; p.N = W.N; p.K = W.K;
  p.epi = c.epi; p.out = c.out; p.ldo = c.ldo; p.resid = c.resid; p.pair_offset = sw ? c.pair_offset : 0;
  p.ntiles = (sw ? c.pair_offset : W.N) / 16;
  p.nblk = W.K / (qb == 4 ? 128 : 64);
  if (c.act == MI_BF16) return qb == 4 ? launch_reg<bf16, 4>(p, sw, st) : launch_reg<bf16, 8>(p, sw, st);
  return qb == 4 ? launch_reg<f16, 4>(p, sw, st) : launch_reg<f16, 8>(p, sw, st);
}

bool gemv_dense_supported(const LinearW& W, const GemvCall& c, size_t rows) {
  static const bool off = getenv("MI_GEMV_DENSE") != nullptr && atoi(getenv("MI_GEMV_DENSE")) == 0;      // (A/B)
  if (off || c.force_v1 || W.layout != 1 || rows < 1 || rows > 8 || c.rnd != RND_NONE || c.kx != 0) return false;
  if (W.lora_b[0] != nullptr || W.lora_b[1] != nullptr || c.out32 || c.silu_cols > 0 || c.glu.kind != GLU_SILU) return false;
  const bool x32 = c.act == MI_F32 && W.wk == WK_BF16;
  if (!x32 && !(W.wk == WK_BF16 && c.act == MI_BF16) && !(W.wk == WK_F16 && c.act == MI_F16)) return false;
  if (c.epi == EPI_SWIGLU_GU8 ? !(x32 && c.pro == PRO_NORM && c.pair_offset % 8 == 0 && W.N == 2 * c.pair_offset)
                              : c.epi != EPI_STORE && c.epi != EPI_STORE_F32 && c.epi != EPI_RESID) return false;
  if (W.K % 64 != 0 || W.N % 16 != 0 || W.K > REG_K) return false;
  // 16-byte loads of x and the norm's weights
  return c.ldx % (x32 ? 4 : 8) == 0 && (uintptr_t)c.x % 16 == 0 && (c.pro != PRO_NORM || (uintptr_t)c.norm_w % 16 == 0);
}

template <typename AT, bool X32>
static int launch_dense(const RegParams& p, bool gu, hipStream_t st) {
  const int grid = std::min(p.ntiles, gemv_cu_count());
  auto go = [&](auto kern) -> int {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), 0, st, p);
    MI_HIP(hipGetLastError());
    return MI_OK;
  };
  if constexpr (X32)
    if (gu) return by_share(p.nblk, 64, [&](auto kw, auto full) { return go(gemv_dense_kernel<AT, X32, true, true, kw.value, full.value>); });
  if (p.norm) return by_share<!X32>(p.nblk, 64, [&](auto kw, auto full) { return go(gemv_dense_kernel<AT, X32, false, true, kw.value, full.value>); });
  return by_share(p.nblk, 64, [&](auto kw, auto full) { return go(gemv_dense_kernel<AT, X32, false, false, kw.value, full.value>); });
}

int launch_gemv_dense(const LinearW& W, const GemvCall& c, size_t rows, hipStream_t st) {
  if (!gemv_dense_supported(W, c, rows)) return fail(MI_ERR_UNSUPPORTED, "gemv_dense: shape / dtype not supported");
  RegParams p{};
  p.x = c.x; p.ldx = c.ldx; p.M = (int)rows;
  p.norm = c.pro == PRO_NORM; p.norm_w = c.norm_w; p.eps = c.eps;
  p.w = W.w; p.N = W.N; p.K = W.K;
  p.epi = c.epi; p.out = c.out; p.ldo = c.ldo; p.resid = c.resid;
  p.ntiles = W.N / 16; p.nblk = W.K / 64;
  const bool gu = c.epi == EPI_SWIGLU_GU8;
  if (c.act == MI_F32) return launch_dense<bf16, true>(p, gu, st);
  return c.act == MI_BF16 ? launch_dense<bf16, false>(p, gu, st) : launch_dense<f16, false>(p, gu, st);
}

// Slices of K: as many as the card has room for beside the tiles, of the same whole pairs of blocks each, and no more than a wave's registers hold.  0: not this kernel
int gemv_side_slices(const LinearW& W, int act, int dim, size_t rows) {
  const bool dense = (W.wk == WK_BF16 && act == MI_BF16) || (W.wk == WK_F16 && act == MI_F16);
  if (!dense || W.layout != 1 || rows < 1 || rows > 8 || dim < 1 || dim > 64 || W.K % 64 != 0 || W.N % 16 != 0 || W.lora_b[0] != nullptr || W.lora_b[1] != nullptr) return 0;
  const int nblk = W.K / 64, tiles = W.N / 16;
  for (int ks = std::max(1, std::min(4, gemv_cu_count() / tiles)); ks <= 4; ++ks)
    if (nblk % ks == 0 && nblk / ks >= 8 && nblk / ks * 64 <= REG_K) return ks;
  return 0;
}

int launch_gemv_side(const LinearW& W, const SideOutCall& c, hipStream_t st) {
  const int ks = gemv_side_slices(W, c.act, c.dim, c.rows);
  if (ks == 0 || c.ldx % 8 != 0 || c.ld % 8 != 0 || c.ld < W.N || ((uintptr_t)c.x | (uintptr_t)c.gate) % 16 != 0) return fail(MI_ERR_UNSUPPORTED, "gemv_side: shape / dtype not supported");
  SideParams p{c.x, c.ldx, c.rows, W.w, W.K / 64, ks, c.resid, c.ld, c.gate, c.dim, c.part, c.z};
  const dim3 grid(W.N / 16, ks);
  auto go = [&](auto kern) -> int {
    hipLaunchKernelGGL(kern, grid, dim3(512), 0, st, p);
    MI_HIP(hipGetLastError());
    return MI_OK;
  };
  if (c.act == MI_BF16) return by_share(p.nblk / ks, 64, [&](auto kw, auto full) { return go(gemv_side_kernel<bf16, kw.value, full.value>); });
  return by_share(p.nblk / ks, 64, [&](auto kw, auto full) { return go(gemv_side_kernel<f16, kw.value, full.value>); });
}

}  // namespace mi
