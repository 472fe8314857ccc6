// misc.hip -- embedding gather, sampler, RoPE tables, small utilities.
#include <algorithm>
#include <type_traits>

#include "kernels.h"

namespace mi {

namespace {

// ------------------------------------------------------------------------------------------
// nn.Embedding / nn.QuantizedEmbedding row gather (llama.py:212, qwen3.py:166).
// Quantised rows are dequantised as round_T(scale*q + bias).
template <typename AT, int WK>
__global__ __launch_bounds__(256) void embed_kernel(LinearW W, EmbedCall c) {
  const int row = blockIdx.x;
  int tok = c.tokens[row];
  tok = min(max(tok, 0), W.N - 1);
  AT* out = (AT*)c.out + (size_t)row * W.K;
  if constexpr (WK == WK_BF16 || WK == WK_F16) {
    // 16-bit tables: 16-byte pieces (8 elements) per thread instead of one element per trip (10 -> ~4 us at the head of every
    // decode step); same values, store_act is applied element by element as below
    if (W.K % 8 == 0) {
      using WT = typename std::conditional<WK == WK_BF16, bf16, f16>::type;
      for (int p8 = threadIdx.x; p8 < W.K / 8; p8 += 256) {
        const char* src = W.layout ? (const char*)W.w + tiled_piece_dense16(tok, p8 * 8, W.K)
                                   : (const char*)W.w + ((size_t)tok * W.K + (size_t)p8 * 8) * 2;
        const uint4 raw = *(const uint4*)src;
        const WT* e = (const WT*)&raw;
        AT o[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = store_act<AT>((float)e[i], c.rnd);
        if constexpr (sizeof(AT) == 2) {
          *(uint4*)(out + (size_t)p8 * 8) = *(const uint4*)o;
        } else {
          *(uint4*)(out + (size_t)p8 * 8) = *(const uint4*)o;
          *(uint4*)(out + (size_t)p8 * 8 + 4) = *(const uint4*)(o + 4);
        }
      }
      return;
    }
  }
  for (int k = threadIdx.x; k < W.K; k += 256) {
    float v;
    const int k8 = k & ~7;
    if constexpr (WK == WK_F32) v = ((const float*)W.w)[(size_t)tok * W.K + k];
    else if constexpr (WK == WK_BF16)
      v = W.layout ? (float)((const bf16*)((const char*)W.w + tiled_piece_dense16(tok, k8, W.K)))[k & 7]
                   : (float)((const bf16*)W.w)[(size_t)tok * W.K + k];
    else if constexpr (WK == WK_F16)
      v = W.layout ? (float)((const f16*)((const char*)W.w + tiled_piece_dense16(tok, k8, W.K)))[k & 7]
                   : (float)((const f16*)W.w)[(size_t)tok * W.K + k];
    else {
      constexpr int BITS = (WK >= WK_Q8_F32) ? 8 : 4;
      constexpr int SDT = (WK - 3) % 3;
      constexpr int PER = 32 / BITS;
      const size_t gi = (size_t)tok * (W.K / W.group) + k / W.group;
      float s, b;
      uint32_t word;
      if (BITS == 4 && SDT != 0 && W.layout) {     // tile-major int4 (repack.hip)
        const char* blk = (const char*)W.w + tiled_block_q4(tok, k, W.K);
        const int so = tiled_q4_scale_off(tok, k);
        if constexpr (SDT == 1) { s = (float)*(const bf16*)(blk + so); b = (float)*(const bf16*)(blk + so + 64); }
        else { s = (float)*(const f16*)(blk + so); b = (float)*(const f16*)(blk + so + 64); }
        word = *(const uint32_t*)(blk + tiled_q4_code_off(tok, k8));
      } else if (BITS == 8 && SDT != 0 && W.layout) {   // tile-major int8
        const char* blk = (const char*)W.w + tiled_block_q8(tok, k, W.K);
        const int so = tiled_q8_scale_off(tok);
        if constexpr (SDT == 1) { s = (float)*(const bf16*)(blk + so); b = (float)*(const bf16*)(blk + so + 32); }
        else { s = (float)*(const f16*)(blk + so); b = (float)*(const f16*)(blk + so + 32); }
        word = *(const uint32_t*)(blk + tiled_q8_code_off(tok, k & ~3));
      } else {
      if constexpr (SDT == 0) { s = ((const float*)W.scales)[gi]; b = ((const float*)W.biases)[gi]; }
      else if constexpr (SDT == 1) { s = (float)((const bf16*)W.scales)[gi]; b = (float)((const bf16*)W.biases)[gi]; }
      else { s = (float)((const f16*)W.scales)[gi]; b = (float)((const f16*)W.biases)[gi]; }
      word = ((const uint32_t*)W.w)[(size_t)tok * (W.K / PER) + k / PER];
      }
      const float q = (float)((word >> (BITS * (k % PER))) & ((1u << BITS) - 1u));
      v = mul_add_unfused(q, s, b);
    }
    out[k] = store_act<AT>(v, c.rnd);
  }
}

template <typename AT>
int launch_embed_wk(const LinearW& W, const EmbedCall& c, hipStream_t st) {
  const dim3 grid(c.rows), block(256);
#define EK(WKV) hipLaunchKernelGGL((embed_kernel<AT, WKV>), grid, block, 0, st, W, c); break
  switch (W.wk) {
    case WK_F32: EK(WK_F32);
    case WK_BF16: EK(WK_BF16);
    case WK_F16: EK(WK_F16);
    case WK_Q4_F32: EK(WK_Q4_F32);
    case WK_Q4_BF16: EK(WK_Q4_BF16);
    case WK_Q4_F16: EK(WK_Q4_F16);
    case WK_Q8_F32: EK(WK_Q8_F32);
    case WK_Q8_BF16: EK(WK_Q8_BF16);
    case WK_Q8_F16: EK(WK_Q8_F16);
    default: return fail(MI_ERR_UNSUPPORTED, "embed: bad weight kind");
  }
#undef EK
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// ------------------------------------------------------------------------------------------
// Sampler: the `sample` closure of generate_step (utils.py:345-364) + top_p_sampling
// (sample_utils.py:3-38).  One 1024-thread workgroup per row; logits stay in L2.
//   greedy: argmax, lowest index among ties (mx.argmax).
//   temp>0: candidates in descending-probability order (ties: ascending id); nucleus keeps the
//           prefix whose INCLUSIVE cumulative probability is <= top_p (empty -> top-1, quirk Q5);
//           the draw is an inverse-CDF pick with one uniform per row.
// Cumulative masses are integers (probability * 2^40 summed with integer atomics), so the
// result does not depend on the order in which threads add.
constexpr int ST = 1024;

// A thread's elements of one row of logits, up to eight at a time: f(values, indices, how many).  A pass is latency-bound if every thread walks it one
// dependent 4-byte load at a time (measured: ~9 us per pass over 32000 logits); 16-byte loads, two in flight per thread (four in flight: no change;
// what bounds the histogram passes is the LDS atomics).
__host__ __device__ __forceinline__ bool row_vec(const float* lg, int V) { return (V & 3) == 0 && (((uintptr_t)lg) & 15) == 0; }
template <class F>
__device__ __forceinline__ void for_row8(const float* lg, int V, F f) {
  if (row_vec(lg, V)) {
    const float4* p4 = (const float4*)lg;
    const int n4 = V >> 2;
    int i = threadIdx.x;
    for (; i + ST < n4; i += 2 * ST) {
      const float4 a = p4[i], b = p4[i + ST];
      const int j = 4 * i, k = 4 * (i + ST);
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      const int at[8] = {j, j + 1, j + 2, j + 3, k, k + 1, k + 2, k + 3};
      f(v, at, std::integral_constant<int, 8>{});
    }
    if (i < n4) {
      const float4 a = p4[i];
      const int j = 4 * i;
      const float v[4] = {a.x, a.y, a.z, a.w};
      const int at[4] = {j, j + 1, j + 2, j + 3};
      f(v, at, std::integral_constant<int, 4>{});
    }
  } else {
    for (int i = threadIdx.x; i < V; i += ST) { const float v[1] = {lg[i]}; const int at[1] = {i}; f(v, at, std::integral_constant<int, 1>{}); }
  }
}
template <class F>
__device__ __forceinline__ void for_row(const float* lg, int V, F f) {
  for_row8(lg, V, [&](const float* v, const int* at, auto n) {
#pragma unroll
    for (int j = 0; j < decltype(n)::value; ++j) f(v[j], at[j]);
  });
}

__device__ __forceinline__ uint32_t order_key(float f) {  // larger float -> larger key
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

struct ArgMax { float v; int i; };
__device__ __forceinline__ ArgMax am_better(ArgMax a, ArgMax b) {
  if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
  return a;
}

__device__ ArgMax block_argmax(ArgMax a, ArgMax* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax b{__shfl_xor(a.v, o, 64), __shfl_xor(a.i, o, 64)};
    a = am_better(a, b);
  }
  __syncthreads();
  if (lane == 0) sh[wave] = a;
  __syncthreads();
  ArgMax r = sh[0];
  for (int w = 1; w < ST / 64; ++w) r = am_better(r, sh[w]);
  return r;
}

__device__ float block_sum(float v, float* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  float r = 0.f;
  for (int w = 0; w < ST / 64; ++w) r += sh[w];
  return r;
}

__device__ __forceinline__ unsigned long long mass_fx(float l, float mx, float inv_t) {
  // exp((l - max)/T) in (0, 1] as 2^40 fixed point
  return (unsigned long long)(__expf((l - mx) * inv_t) * 1099511627776.0f);
}

// the cumulative mass that the pick exceeds
__device__ __forceinline__ unsigned long long pick_mass(float u, unsigned long long kept) {
  const unsigned long long y = (unsigned long long)((double)u * (double)kept);
  return kept > 0 && y >= kept ? kept - 1 : y;
}

// Philox-4x32-10 (key = seed, counter = (step, row)) -> one uniform in [0,1)
__device__ float philox_uniform(uint64_t seed, uint64_t step, uint32_t row) {
  uint32_t c0 = (uint32_t)step, c1 = (uint32_t)(step >> 32), c2 = row, c3 = 0x9E3779B9u;
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0, n1 = (uint32_t)p1;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1, n3 = (uint32_t)p0;
    c0 = n0; c1 = n1; c2 = n2; c3 = n3;
    k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
  }
  return (float)(c0 >> 8) * (1.0f / 16777216.0f);
}

// Find the descending-order prefix whose cumulative mass is <= target.
// Returns (through sh_*) the key of the first element NOT wholly inside the prefix (`kstar`),
// how many elements with key == kstar are inside the prefix (`ntie`), and the prefix mass.
// `limit_key/limit_tie`: only elements in a previously selected prefix are considered
// (key > limit_key, or key == limit_key and tie-rank < limit_tie); pass limit_key = 0,
// limit_tie = INT_MAX for "all".
struct Prefix { uint32_t kstar; int ntie; unsigned long long mass; int count; };

// Level-0 histogram (top 8 key bits) of the whole row, built once per row and shared by every descent.  The logits of
// one row share a few exponents, i.e. a few level-0 bins: the adds are spread over 8 private copies (by lane) to cut
// the same-address serialisation of the LDS atomics, then folded.
struct Hist0 { unsigned long long m[256]; int c[256]; };

__device__ void build_hist0(const float* lg, int V, float mx, float inv_t, unsigned long long (*pm)[8], int (*pc)[8],
                            Hist0* h0) {
  // [bin][copy]: the 8 copies of a bin are neighbours, i.e. on different LDS banks ([copy][bin] would put them 2 KiB
  // apart -- all on one bank)
  for (int i = threadIdx.x; i < 8 * 256; i += ST) { pm[i >> 3][i & 7] = 0; pc[i >> 3][i & 7] = 0; }
  __syncthreads();
  const int cp = threadIdx.x & 7;
  for_row(lg, V, [&](float l, int) {
    const int bin = order_key(l) >> 24;
    atomicAdd(&pm[bin][cp], mass_fx(l, mx, inv_t));
    atomicAdd(&pc[bin][cp], 1);
  });
  __syncthreads();
  if (threadIdx.x < 256) {
    unsigned long long m = 0; int n = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) { m += pm[threadIdx.x][k]; n += pc[threadIdx.x][k]; }
    h0->m[threadIdx.x] = m; h0->c[threadIdx.x] = n;
  }
  __syncthreads();
}

// Which bin holds the element at which the descending cumulative mass (starting from `above`) first exceeds
// `target`?  One wave scans the 256 bins from 255 down (4 bins per lane + a wave scan: two block barriers instead of
// a block-wide scan); returns through out_sh: mass / count of everything above that bin, and the bin (-1: all fits).
__device__ void select_bin(const unsigned long long* hist_m, const int* hist_c, unsigned long long above, int above_cnt,
                           unsigned long long target, Prefix* out_sh) {
  __syncthreads();
  if (threadIdx.x < 64) {
    const int L = threadIdx.x;
    unsigned long long m[4], tm = 0; int c[4], tc = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) { m[j] = hist_m[255 - (4 * L + j)]; c[j] = hist_c[255 - (4 * L + j)]; tm += m[j]; tc += c[j]; }
    unsigned long long im = tm; int ic = tc;                       // inclusive scan over lanes = descending bins
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned long long om = __shfl_up(im, off, 64);
      const int oc = __shfl_up(ic, off, 64);
      if (L >= off) { im += om; ic += oc; }
    }
    unsigned long long cum = above + im - tm; int cnt = above_cnt + ic - tc;
    int pos = 256; unsigned long long pm = 0; int pc = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (pos == 256) {
        if (c[j] > 0 && cum + m[j] > target) { pos = 4 * L + j; pm = cum; pc = cnt; }
        else { cum += m[j]; cnt += c[j]; }
      }
    }
    int best = pos;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = min(best, __shfl_xor(best, o, 64));
    if (best == 256) { if (L == 63) { out_sh->mass = cum; out_sh->count = cnt; out_sh->ntie = -1; } }
    else if (pos == best) { out_sh->mass = pm; out_sh->count = pc; out_sh->ntie = 255 - best; }
  }
  __syncthreads();
}

// Find the descending-order prefix whose cumulative mass is <= target (radix descent over the order key, 8 bits per
// level; level 0 comes from the cached histogram, the lower levels touch only the elements under the chosen prefix).
// KERNEL: a function for each kernel that calls it, so that it knows the places in LDS (one for both: top-p of 50257 logits 111 us, 106 with its own)
template <int KERNEL>
__device__ Prefix find_prefix(const float* lg, int V, float mx, float inv_t, unsigned long long target,
                              unsigned long long* hist_m, int* hist_c, Prefix* out_sh, const Hist0* h0) {
  uint32_t prefix_bits = 0;   // fixed high bits of kstar so far
  uint32_t prefix_mask = 0;
  unsigned long long above = 0;  // mass of keys strictly greater than the current candidate bin
  int above_cnt = 0;
  for (int level = 0; level < 4; ++level) {
    const int shift = 24 - 8 * level;
    if (level == 0) {
      select_bin(h0->m, h0->c, above, above_cnt, target, out_sh);
    } else {
      __syncthreads();
      for (int i = threadIdx.x; i < 256; i += ST) { hist_m[i] = 0; hist_c[i] = 0; }
      __syncthreads();
      for_row(lg, V, [&](float l, int) {
        const uint32_t k = order_key(l);
        if ((k & prefix_mask) == prefix_bits) {
          const int bin = (k >> shift) & 255;
          atomicAdd(&hist_m[bin], mass_fx(l, mx, inv_t));
          atomicAdd(&hist_c[bin], 1);
        }
      });
      __syncthreads();
      select_bin(hist_m, hist_c, above, above_cnt, target, out_sh);
    }
    above = out_sh->mass;
    above_cnt = out_sh->count;
    const int bin = out_sh->ntie;
    if (bin < 0) {
      __syncthreads();
      Prefix r{0u, 0, above, above_cnt};
      return r;  // the whole (sub)set is inside the prefix
    }
    prefix_bits |= (uint32_t)bin << shift;
    prefix_mask |= 255u << shift;
  }
  // kstar = prefix_bits: all elements with this exact key have the same mass; count how many fit
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long each = mass_fx(__uint_as_float((prefix_bits & 0x80000000u) ? (prefix_bits & 0x7fffffffu) : ~prefix_bits), mx, inv_t);
    unsigned long long cum = above;
    int n = 0;
    while (each > 0 && cum + each <= target) { cum += each; ++n; }
    out_sh->mass = cum;
    out_sh->ntie = n;
    out_sh->count = above_cnt + n;
  }
  __syncthreads();
  Prefix r{prefix_bits, out_sh->ntie, out_sh->mass, out_sh->count};
  __syncthreads();
  return r;
}

// index of the (rank)-th smallest token id among those whose key == kstar.
// 16-bit logits make big tie groups (hundreds of ids share one value), so rank can be large: ONE counting pass
// in index order (chunks of 4 * ST ids, thread t of chunk j owns ids 4 * (ST * j + t) .. + 3; per-(chunk, wave)
// tie counts via ballots), a scan of that small table, and the owning wave finds the id among its 256.
constexpr int TIE_TBL = 1024;       // (chunk, wave) entries: V <= 4 * ST * (TIE_TBL / 16) = 262144 ids
__device__ int nth_tie(const float* lg, int V, uint32_t kstar, int rank, int* sh_i, int* tbl, int* found) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nch = (V + 4 * ST - 1) / (4 * ST);
  const bool vec = (V & 3) == 0 && (((uintptr_t)lg) & 15) == 0 && nch * (ST / 64) <= TIE_TBL;
  if (vec) {
    auto ties_of = [&](int j, bool (&is)[4]) {
      const int base = 4 * (ST * j + (int)threadIdx.x);
      float4 v = {0.f, 0.f, 0.f, 0.f};
      if (base < V) v = *(const float4*)(lg + base);
      is[0] = base < V && order_key(v.x) == kstar; is[1] = base < V && order_key(v.y) == kstar;
      is[2] = base < V && order_key(v.z) == kstar; is[3] = base < V && order_key(v.w) == kstar;
    };
    for (int j = 0; j < nch; ++j) {
      bool is[4];
      ties_of(j, is);
      int n = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) n += __popcll(__ballot(is[e]));
      if (lane == 0) tbl[j * (ST / 64) + wave] = n;
    }
    if (threadIdx.x == 0) *found = -1;
    __syncthreads();
    if (threadIdx.x == 0) {                       // (chunk, wave) that holds the rank-th tie, and the rank inside it
      int left = rank, at = -1;
      for (int i = 0; i < nch * (ST / 64); ++i) {
        const int n = tbl[i];
        if (left < n) { at = i; break; }
        left -= n;
      }
      sh_i[0] = at; sh_i[1] = left;
    }
    __syncthreads();
    const int at = sh_i[0], left = sh_i[1];
    if (at >= 0 && wave == at % (ST / 64)) {
      bool is[4];
      ties_of(at / (ST / 64), is);
      const unsigned long long lt = (1ull << lane) - 1ull;
      int before = 0, own = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) { before += __popcll(__ballot(is[e]) & lt); own += is[e] ? 1 : 0; }
      if (left >= before && left < before + own) {
        int k = left - before;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (is[e]) { if (k == 0) *found = 4 * (ST * (at / (ST / 64)) + (int)threadIdx.x) + e; --k; }
      }
    }
    __syncthreads();
    const int r = *found;
    __syncthreads();
    return r;                                     // -1: fewer than rank + 1 ties (the caller falls back to the arg-max)
  }
  int last = -1;
  for (int r = 0; r <= rank; ++r) {
    int best = 0x7fffffff;
    for_row(lg, V, [&](float l, int i) {
      if (i > last && i < best && order_key(l) == kstar) best = i;
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = min(best, __shfl_xor(best, o, 64));
    __syncthreads();
    if (lane == 0) sh_i[wave] = best;
    __syncthreads();
    best = sh_i[0];
    for (int w = 1; w < ST / 64; ++w) best = min(best, sh_i[w]);
    last = best;
    __syncthreads();
  }
  return last;
}

// LDS of a draw
struct DrawLds {
  unsigned long long* hist_m; int* hist_c; Prefix* p; unsigned long long (*priv_m)[8]; int (*priv_c)[8]; Hist0* h0; int* tie_tbl; int* i; int* sel;
};

// The draw at temperature 1 / inv_t by one workgroup that walks the row once per level of the descents; `best` if nothing can be drawn
template <int KERNEL>
__device__ __forceinline__ int draw_row(const float* lg, int V, float mx, float inv_t, float top_p, float u, int best, const DrawLds& s) {
  // total mass Z (integer) = sum of the level-0 histogram, which every descent below reuses
  build_hist0(lg, V, mx, inv_t, s.priv_m, s.priv_c, s.h0);
  select_bin(s.h0->m, s.h0->c, 0ull, 0, ~0ull, s.p);       // target = +inf: everything fits
  Prefix all{0u, 0, s.p->mass, s.p->count};
  const unsigned long long Z = all.mass;
  Prefix kept = all;
  uint32_t keep_key = 0; int keep_tie = 0x7fffffff;
  if (top_p > 0.f && top_p < 1.f) {
    const unsigned long long tgt = (unsigned long long)((double)top_p * (double)Z);
    kept = find_prefix<KERNEL>(lg, V, mx, inv_t, tgt, s.hist_m, s.hist_c, s.p, s.h0);
    keep_key = kept.kstar; keep_tie = kept.ntie;
    if (kept.count == 0) {  // top token alone exceeds top_p (reference: 0/0); keep top-1
      kept.count = 1; kept.mass = mass_fx(mx, mx, inv_t);
      keep_key = order_key(mx); keep_tie = 1;
    }
  }
  // first candidate whose inclusive cumulative mass exceeds u * Z_kept
  const unsigned long long y = pick_mass(u, kept.mass);
  Prefix pk = find_prefix<KERNEL>(lg, V, mx, inv_t, y, s.hist_m, s.hist_c, s.p, s.h0);
  // pk.count candidates lie strictly before the pick; the pick is the next one in order
  int rank_in_key = pk.ntie;
  uint32_t key = pk.kstar;
  if (pk.count >= kept.count) {  // numerical corner: clamp to the last kept candidate
    key = keep_key; rank_in_key = max(keep_tie - 1, 0);
    if (keep_tie == 0x7fffffff) { key = pk.kstar; rank_in_key = max(pk.ntie - 1, 0); }
  }
  const int token = nth_tie(lg, V, key, rank_in_key, s.i, s.tie_tbl, s.sel);
  return token < 0 || token >= V ? best : token;
}

__device__ __forceinline__ void add_bias(const SampleCall& c, float* lg, int lo, int hi) {      // logits[:, indices] += values (utils.py:346-349)
  for (int i = threadIdx.x; i < c.n_bias; i += ST) {
    const int id = c.bias_ids[i];
    if (id >= lo && id < hi) lg[id] = round_rt(lg[id] + c.bias_vals[i], c.rnd);
  }
  __syncthreads();
}

// max / argmax and the sum of exp: one walk, a thread's sum relative to its own maximum so far
struct MaxSum {
  ArgMax best{-INFINITY, 0x7fffffff};
  float part = 0.f;
  template <class N>
  __device__ __forceinline__ void operator()(const float* l, const int* idx, N) {
    const float was = best.v;
#pragma unroll
    for (int j = 0; j < N::value; ++j) best = am_better(best, ArgMax{l[j], idx[j]});
    if (best.v > was) part *= __expf(was - best.v);
    const float ref = best.v == -INFINITY ? 0.f : best.v;
#pragma unroll
    for (int j = 0; j < N::value; ++j) part += __expf(l[j] - ref);
  }
};

__global__ __launch_bounds__(ST) void sample_kernel(SampleCall c) {
  __shared__ ArgMax sh_am[ST / 64];
  __shared__ float sh_f[ST / 64];
  __shared__ int sh_i[ST / 64];
  __shared__ unsigned long long hist_m[256];
  __shared__ int hist_c[256];
  __shared__ Prefix sh_p;
  __shared__ unsigned long long priv_m[256][8];
  __shared__ int priv_c[256][8], sel_sh;
  __shared__ Hist0 h0;
  __shared__ int tie_tbl[TIE_TBL];
  const DrawLds sh_d{hist_m, hist_c, &sh_p, priv_m, priv_c, &h0, tie_tbl, sh_i, &sel_sh};
  const int b = blockIdx.x, V = c.V;
  float* lg = c.logits + (size_t)b * V;
  // per-row sampling parameters (continuous batching: every request keeps its own) or the call's scalars
  const float temperature = c.row_temp ? c.row_temp[b] : c.temperature;
  const float top_p = c.row_top_p ? c.row_top_p[b] : c.top_p;

  if (c.n_bias > 0) add_bias(c, lg, 0, V);
  MaxSum take;
  for_row8(lg, V, [&](const float* l, const int* idx, auto n) { take(l, idx, n); });
  ArgMax& mine = take.best;
  ArgMax a = block_argmax(mine, sh_am);
  const float mx = a.v;
  const float se = block_sum(mine.v == -INFINITY ? take.part : take.part * __expf(mine.v - mx), sh_f);
  const float lse = mx + __logf(se);
  if (threadIdx.x == 0 && c.row_stats) { c.row_stats[2 * b] = mx; c.row_stats[2 * b + 1] = lse; }

  int token = a.i;
  const int forced = c.forced ? c.forced[b] : 0;
  if (c.forced) {
    if (forced >= 0 && forced < V) token = forced;
  } else if (temperature != 0.f) {
    const float u = c.uniforms ? c.uniforms[b] : philox_uniform(c.seed, c.step, (uint32_t)b);
    token = draw_row<0>(lg, V, mx, 1.0f / temperature, top_p, u, a.i, sh_d);
  }
  // logprobs are reported as (lg - mx) * lp_scale - lp_lse: the plain log-softmax, or the one of logits / T
  float lp_scale = 1.0f, lp_lse = lse - mx;
  if (c.lp_temp && temperature > 0.f) {
    lp_scale = 1.0f / temperature;
    float st = se;                               // T = 1: the sum of the walk above (no second one)
    if (lp_scale != 1.0f) {                      // (uniform)
      st = 0.f;
      for_row(lg, V, [&](float l, int) { st += __expf((l - mx) * lp_scale); });
      st = block_sum(st, sh_f);
    }
    lp_lse = __logf(st);
  }
  // a row without a single comparable logit (all NaN / -inf: a broken checkpoint, an overflow upstream) has no
  // arg-max; it yields token 0 rather than an id that the next kernels would use as an address
  if (token < 0 || token >= V) token = 0;
  if (threadIdx.x == 0) {
    c.tokens_out[b] = token;
    if (c.logprob_out) c.logprob_out[b] = (c.forced && forced < 0) ? 0.f : (lg[token] - mx) * lp_scale - lp_lse;
  }
  // ---- top-k logprobs: k rounds of arg-max over the threads' best remaining elements; the winner's wave looks for its next one
  const bool vec = row_vec(lg, V);
  for (int r = 0; r < c.top_logprobs; ++r) {
    const ArgMax t = block_argmax(mine, sh_am);
    if (threadIdx.x == 0) {
      c.topk_ids[(size_t)b * c.top_logprobs + r] = t.i < V ? t.i : 0;
      c.topk_logprobs[(size_t)b * c.top_logprobs + r] = (t.v - mx) * lp_scale - lp_lse;
    }
    if (t.i >= V || r + 1 == c.top_logprobs) continue;            // (uniform)
    const int owner = (vec ? t.i >> 2 : t.i) % ST;
    if ((int)threadIdx.x >> 6 != owner >> 6) continue;
    ArgMax best{-INFINITY, 0x7fffffff};
    const auto next = [&](float v, int i) { if (v < t.v || (v == t.v && i > t.i)) best = am_better(best, ArgMax{v, i}); };
    for (int i = owner + (threadIdx.x & 63) * ST; i < (vec ? V >> 2 : V); i += 64 * ST) {
      if (vec) {
        const float4 q = ((const float4*)lg)[i];
        next(q.x, 4 * i); next(q.y, 4 * i + 1); next(q.z, 4 * i + 2); next(q.w, 4 * i + 3);
      } else next(lg[i], i);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = am_better(best, ArgMax{__shfl_xor(best.v, o, 64), __shfl_xor(best.i, o, 64)});
    if ((int)threadIdx.x == owner) mine = best;
  }
}

// ---- the same over several workgroups a row ------------------------------------------------------------------------------
// One workgroup per row leaves the card idle at a decode step's few rows and is bound by its own walks of the row, four to eight of them in a draw, each a
// chain of loads, LDS atomics and barriers.  Here up to SG workgroups take a row's parts, in two launches (greedy, forced) or three:
//   sample_parts:  maximum and sum of exp of every part, the best element of every 16 threads' share
//   sample_masses: masses of every part in SNB bins of (max - l) / T from 0 to where the row's elements end, at most 28: beyond, a mass is 0
//   sample_draw:   the bins hold the cut of the nucleus and the pick in known bins; their elements are collected, the last workgroup of the row to arrive
//                  sorts them (key, id) and finds both, exactly: the integer masses add up to the same whatever the order.  One more workgroup does the
//                  most likely tokens.  Probabilities of row 0 are made here: no launch of their own.
// A row with NaN or +inf, a temperature that is no positive number, or more than SCAP elements in those bins (thousands of equal logits) is drawn by
// draw_row, the launches in front for nothing (8 rows of 128256 210 us, 172 by one workgroup a row).  us, one workgroup per row / here: 8 rows of 32000 logits top-p with 5 log-probabilities 70 / 35, temperature alone 44 / 30, greedy with 5 23 / 19;
// 128256 logits 176 / 57, 128 / 41, 32 / 22, greedy 20 / 15; 64 rows of 128256 194 / 70, greedy 20.5 / 18.8; 512 rows top-p 454 / 306; 256 rows of 16384 56 / 59.
// Greedy without them: 32000 logits 11 / 11, 64 rows of 50304 13.0 / 14.5, 128 rows of 128256 21 / 24.  What is left of a draw is its chain: three launches,
// the sum of the bins (3 us), the list through memory (4), the sort (3 to 6).
constexpr int SG = SAMPLE_PARTS, SNB = 2048, SCAP = 4096, SW = ST / 64, SLABS = ST / 16;
struct SampleRow {
  float pmax[SG], psum[SG], psum_t[SG], scale;
  int pidx[SG], odd[SG];
  unsigned listed, arrived;
  alignas(16) unsigned long long list[SCAP];         // order key << 32 | ~id: descending order is the candidates' order
  ArgMax slab[SG * SLABS];
};
// part g of a row: float4 pieces [first, last)
__device__ __forceinline__ int part_at(int V, int g, int np) { return (int)((long)(V >> 2) * g / np); }
template <class F>
__device__ __forceinline__ void for_part(const float* lg, int lo, int hi, F f) {
  const float4* p4 = (const float4*)lg;
  int i = lo + threadIdx.x;
  for (; i + 3 * ST < hi; i += 4 * ST) {
    float4 q[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) q[j] = p4[i + j * ST];
#pragma unroll
    for (int j = 0; j < 4; ++j) f(q[j], 4 * (i + j * ST));
  }
  for (; i < hi; i += ST) f(p4[i], 4 * i);
}

struct RowHead { float mx, se, lse; int best; bool odd; };
// the np parts of a row together, in their order: the same in every workgroup
__device__ __forceinline__ RowHead row_head(const SampleRow* w, int np) {
  RowHead h;
  ArgMax a{-INFINITY, 0x7fffffff};
  h.odd = false;
#pragma unroll
  for (int g = 0; g < SG; ++g) {                  // (a part beyond the last is the last once more: loads, no branches)
    const int k = min(g, np - 1);
    a = am_better(a, ArgMax{w->pmax[k], w->pidx[k]}); h.odd |= w->odd[k] != 0;
  }
  h.mx = a.v; h.best = a.i; h.se = 0.f;
#pragma unroll
  for (int g = 0; g < SG; ++g) {
    const int k = min(g, np - 1);
    const float t = w->pmax[k] == -INFINITY ? w->psum[k] : w->psum[k] * __expf(w->pmax[k] - a.v);
    h.se += g < np ? t : 0.f;
  }
  h.lse = a.v + __logf(h.se);
  return h;
}

// Bins per unit of max - l.  Any number is right -- what lies beyond is in the last bin --, as long as both kernels use the same.  The range: three times the distance from the maximum to
// the logarithm of the mean exp(l): all of a bell (that distance is 4.5 deviations less half a square).  28 T of every row, 73 bins a unit, left 600 elements of 128256 of deviation 1.3 in a bin
// at the cut, and of rows that T makes flat more than a list takes: deviation 1, top-p, 8 rows at T = 1 / 5 / 20 67 / 201 / 203 us (one workgroup a row 169 / 172 / 173), 47 at all three now.
__device__ __forceinline__ float bin_scale(const RowHead& h, int V, float inv_t) {
  const float range = 3.0f * inv_t * (__logf((float)V) - (h.lse - h.mx));
  return inv_t * SNB * __builtin_amdgcn_rcpf(fminf(fmaxf(range, 1e-30f), 28.0f));
}
__device__ __forceinline__ int mass_bin(float l, float mx, float scale) { return (int)fminf((mx - l) * scale, SNB - 1); }

__global__ __launch_bounds__(ST) void sample_parts_kernel(SampleCall c, SampleRow* ws) {
  __shared__ ArgMax sh_am[SW];
  __shared__ float sh_f[SW];
  const int g = blockIdx.x, b = blockIdx.y, V = c.V, lo = part_at(V, g, gridDim.x), hi = part_at(V, g + 1, gridDim.x);
  float* lg = c.logits + (size_t)b * V;
  SampleRow* w = ws + b;
  if (c.n_bias > 0) add_bias(c, lg, 4 * lo, 4 * hi);
  MaxSum take;
  bool odd = false;
  for_part(lg, lo, hi, [&](float4 q, int at) {
    const float v[4] = {q.x, q.y, q.z, q.w};
    const int ids[4] = {at, at + 1, at + 2, at + 3};
    take(v, ids, std::integral_constant<int, 4>{});
#pragma unroll
    for (int j = 0; j < 4; ++j) odd |= !(v[j] < INFINITY);
  });
  ArgMax t = take.best;
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) t = am_better(t, ArgMax{__shfl_xor(t.v, o, 64), __shfl_xor(t.i, o, 64)});
  if ((threadIdx.x & 15) == 0) w->slab[g * SLABS + (threadIdx.x >> 4)] = t;
  const ArgMax a = block_argmax(take.best, sh_am);
  const float se = block_sum(take.best.v == -INFINITY ? take.part : take.part * __expf(take.best.v - a.v), sh_f);
  odd = __syncthreads_or(odd);
  if (threadIdx.x == 0) {
    w->pmax[g] = a.v; w->pidx[g] = a.i; w->psum[g] = se; w->odd[g] = odd;
    if (g == 0) { w->listed = 0; w->arrived = 0; }
  }
}

__global__ __launch_bounds__(ST) void sample_masses_kernel(SampleCall c, SampleRow* ws, unsigned long long* hist) {
  __shared__ unsigned long long m[SNB];
  __shared__ float sh_f[SW];
  const int g = blockIdx.x, b = blockIdx.y, V = c.V;
  const float* lg = c.logits + (size_t)b * V;
  SampleRow* w = ws + b;
  const float temperature = c.row_temp ? c.row_temp[b] : c.temperature;
  if (!(temperature > 0.f)) return;
  const int np = gridDim.x;
  const RowHead h = row_head(w, np);
  const float inv_t = 1.0f / temperature, scale = bin_scale(h, V, inv_t);
  if (g == 0 && threadIdx.x == 0) w->scale = scale;
  for (int i = threadIdx.x; i < SNB; i += ST) m[i] = 0;
  __syncthreads();
  float st = 0.f;
  for_part(lg, part_at(V, g, np), part_at(V, g + 1, np), [&](float4 q, int) {
    const float v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned long long each = mass_fx(v[j], h.mx, inv_t);
      if (each > 0 && !h.odd) atomicAdd(&m[mass_bin(v[j], h.mx, scale)], each);
      if (c.lp_temp) st += __expf((v[j] - h.mx) * inv_t);
    }
  });
  if (c.lp_temp) {                               // (uniform)
    st = block_sum(st, sh_f);
    if (threadIdx.x == 0) w->psum_t[g] = st;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < SNB; i += ST) hist[((size_t)b * np + g) * SNB + i] = m[i];
}

// inclusive sum over the workgroup's threads; `sh`: a word per wave
__device__ __forceinline__ unsigned long long block_scan(unsigned long long v, unsigned long long* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  __syncthreads();
  if (lane == 63) sh[wave] = v;
  __syncthreads();
  for (int k = 0; k < wave; ++k) v += sh[k];
  return v;
}

// Descending sort of E ST words, word e ST + t in thread t's a[e]: exchanges below 64 places inside a wave, from ST on inside a thread, between through LDS.
// n: a power of two from 64 on; the words behind the first n stay where they are.
template <int E>
__device__ __forceinline__ void sort_desc(unsigned long long (&a)[E], int n, unsigned long long* sh) {
  const int tid = threadIdx.x;
  for (int k = 2; k <= n; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (j >= ST) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int o = e ^ (j / ST);
          if (o > e && o < E) {
            const unsigned long long x = a[e], y = a[o < E ? o : e];
            const bool swap = ((e * ST + tid) & k) == 0 ? x < y : x > y;
            a[e] = swap ? y : x; a[o < E ? o : e] = swap ? x : y;
          }
        }
        continue;
      }
      if (j >= 64) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) sh[e * ST + tid] = a[e];
        __syncthreads();
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = e * ST + tid;
        if (i >= n) continue;                                      // (whole waves)
        const unsigned long long x = a[e], y = j >= 64 ? sh[i ^ j] : __shfl_xor(x, j, 64);
        const bool first = (i & j) == 0, down = (i & k) == 0;      // the first of a pair keeps the larger word where the run descends
        a[e] = (first == down) == (x < y) ? y : x;
      }
    }
}

struct DrawPlan { unsigned long long tgt, cut_above, pick_above; int cut, p0, p1; bool nucleus; float u, inv_t, mx, scale; };

// The pick among the row's n collected words
template <int E>
__device__ int pick_listed(const SampleRow* w, int n, const DrawPlan& d, unsigned long long* buf, unsigned long long* scan, int* found) {
  const int tid = threadIdx.x;
  unsigned long long a[E];
#pragma unroll
  for (int e = 0; e < E; ++e) a[e] = e * ST + tid < n ? __hip_atomic_load(&w->list[e * ST + tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
  int n2 = 64;
  while (n2 < n) n2 <<= 1;
  sort_desc<E>(a, n2, buf);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) buf[e * ST + tid] = a[e];
  __syncthreads();
  // now words [E tid, E tid + E) of the order
  unsigned long long m[E];
  int bin[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = E * tid + e;
    a[e] = buf[i];
    const uint32_t k = (uint32_t)(a[e] >> 32);
    const float l = __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
    m[e] = i < n ? mass_fx(l, d.mx, d.inv_t) : 0ull;
    bin[e] = i < n ? mass_bin(l, d.mx, d.scale) : -1;
  }
  unsigned long long kept = d.tgt;               // (no nucleus: everything, and tgt is the whole mass)
  if (d.nucleus) {
    unsigned long long own = 0, in = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) own += bin[e] == d.cut ? m[e] : 0ull;
    unsigned long long cum = d.cut_above + block_scan(own, scan) - own;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (bin[e] == d.cut && cum + m[e] <= d.tgt) { cum += m[e]; in += m[e]; }
      else if (bin[e] == d.cut) cum = ~0ull >> 1;          // (behind the first that does not fit nothing does)
    // (a thread in front of the one that holds the first misfit has all its words in, one behind none: cum is past the target already)
    __syncthreads();
    const unsigned long long incl = block_scan(in, scan);
    __syncthreads();
    if (tid == ST - 1) scan[SW] = incl;
    __syncthreads();
    kept = d.cut_above + scan[SW];
    if (kept == 0) kept = mass_fx(d.mx, d.mx, d.inv_t);    // top token alone exceeds top_p (reference: 0/0); keep top-1
  }
  const unsigned long long y = pick_mass(d.u, kept);
  unsigned long long own = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) own += bin[e] >= d.p0 && bin[e] <= d.p1 ? m[e] : 0ull;
  unsigned long long cum = d.pick_above + block_scan(own, scan) - own;
  if (tid == 0) *found = 0x7fffffff;
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (bin[e] < d.p0 || bin[e] > d.p1) continue;
    if (cum <= y && cum + m[e] > y) atomicMin(found, (int)(0xffffffffu - (uint32_t)a[e]));
    cum += m[e];
  }
  __syncthreads();
  const int r = *found;
  __syncthreads();
  return r;
}

// np: parts of a row.  gridDim.x: nwg workgroups for the row (one where nothing is drawn), and one more for the most likely tokens
__global__ __launch_bounds__(ST) void sample_draw_kernel(SampleCall c, SampleRow* ws, const unsigned long long* hist, int np, int nwg) {
  __shared__ union {
    struct { unsigned long long priv_m[256][8], hist_m[256]; Hist0 h0; int priv_c[256][8], hist_c[256], tie_tbl[TIE_TBL], i[SW], sel; Prefix p; } d;
    unsigned long long buf[SCAP];
  } sh;
  __shared__ unsigned long long scan[SW + 1];
  __shared__ unsigned long long bin_hi[SNB];
  __shared__ int sel[4];
  __shared__ unsigned base_sh;
  const DrawLds sh_d{sh.d.hist_m, sh.d.hist_c, &sh.d.p, sh.d.priv_m, sh.d.priv_c, &sh.d.h0, sh.d.tie_tbl, sh.d.i, &sh.d.sel};
  const int g = blockIdx.x, b = blockIdx.y, V = c.V, tid = threadIdx.x;
  const float* lg = c.logits + (size_t)b * V;
  SampleRow* w = ws + b;
  const float temperature = c.row_temp ? c.row_temp[b] : c.temperature;
  const bool draws = c.forced == nullptr && temperature != 0.f;
  if (g < nwg && g > 0 && !draws) return;
  const RowHead h = row_head(w, np);
  const float mx = h.mx;
  float lp_scale = 1.0f, lp_lse = h.lse - mx;    // logprobs are reported as (lg - mx) * lp_scale - lp_lse
  if (c.lp_temp && temperature > 0.f) {
    lp_scale = 1.0f / temperature;
    float st = h.se;
    if (lp_scale != 1.0f) {
      st = 0.f;
#pragma unroll
      for (int k = 0; k < SG; ++k)
        if (k < np) st += w->psum_t[k];
    }
    lp_lse = __logf(st);
  }
  if (g == nwg) {                                // the k most likely: one wave, a share of 16 threads in each of np lanes' registers; the winner's is read again
    if (tid >= 64) return;
    static_assert(SLABS == 64, "a lane per share of a part");
    ArgMax best[SG];
#pragma unroll
    for (int i = 0; i < SG; ++i) {
      best[i] = w->slab[min(i, np - 1) * SLABS + tid];
      if (i >= np) best[i] = ArgMax{-INFINITY, 0x7fffffff};
    }
    for (int r = 0; r < c.top_logprobs; ++r) {
      ArgMax t = best[0];
      int at = 0;
#pragma unroll
      for (int i = 1; i < SG; ++i) {
        const ArgMax n = am_better(t, best[i]);
        if (n.i != t.i) { t = n; at = i; }
      }
      at = at * SLABS + tid;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const ArgMax n{__shfl_xor(t.v, o, 64), __shfl_xor(t.i, o, 64)};
        const int na = __shfl_xor(at, o, 64);
        if (n.v > t.v || (n.v == t.v && n.i < t.i)) { t = n; at = na; }
      }
      if (tid == 0) {
        c.topk_ids[(size_t)b * c.top_logprobs + r] = t.i < V ? t.i : 0;
        c.topk_logprobs[(size_t)b * c.top_logprobs + r] = (t.v - mx) * lp_scale - lp_lse;
      }
      if (t.i >= V || r + 1 == c.top_logprobs) continue;          // (uniform)
      ArgMax next{-INFINITY, 0x7fffffff};
      const int part = at / SLABS, hi = part_at(V, part + 1, np);
      auto look = [&](float4 q, int i) {
        const float v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (v[j] < t.v || (v[j] == t.v && 4 * i + j > t.i)) next = am_better(next, ArgMax{v[j], 4 * i + j});
      };
      int i = part_at(V, part, np) + at % SLABS * 16 + (tid & 15) + (tid >> 4) * ST;      // the share's pieces are ST apart: four of them a trip, or 16
      for (; i + 12 * ST < hi; i += 16 * ST) {
        float4 q[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = ((const float4*)lg)[i + 4 * j * ST];
#pragma unroll
        for (int j = 0; j < 4; ++j) look(q[j], i + 4 * j * ST);
      }
      for (; i < hi; i += 4 * ST) look(((const float4*)lg)[i], i);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) next = am_better(next, ArgMax{__shfl_xor(next.v, o, 64), __shfl_xor(next.i, o, 64)});
#pragma unroll
      for (int k = 0; k < SG; ++k)
        if (at == k * SLABS + tid) best[k] = next;
    }
    return;
  }
  int token = h.best;
  const int forced = c.forced ? c.forced[b] : 0;
  if (c.forced) {
    if (forced >= 0 && forced < V) token = forced;
  } else if (draws) {
    const float inv_t = 1.0f / temperature;
    const float top_p = c.row_top_p ? c.row_top_p[b] : c.top_p;
    const float u = c.uniforms ? c.uniforms[b] : philox_uniform(c.seed, c.step, (uint32_t)b);
    if (h.odd || !(mx > -INFINITY) || !(temperature > 0.f) || !(inv_t < INFINITY)) {      // (uniform)
      if (g > 0) return;
      token = draw_row<1>(lg, V, mx, inv_t, top_p, u, h.best, sh_d);
    } else {
      DrawPlan d;
      d.u = u; d.inv_t = inv_t; d.mx = mx; d.scale = w->scale;
      d.nucleus = top_p > 0.f && top_p < 1.f;
      unsigned long long lower = 0, own = 0;     // (two bins a thread)
#pragma unroll
      for (int k = 0; k < SG; ++k) {
        const ulonglong2 m = ((const ulonglong2*)(hist + ((size_t)b * np + min(k, np - 1)) * SNB))[tid];
        lower += k < np ? m.x : 0ull; own += k < np ? m.x + m.y : 0ull;
      }
      const unsigned long long incl = block_scan(own, scan), first = incl - own + lower;
      bin_hi[2 * tid] = first;
      bin_hi[2 * tid + 1] = incl;
      if (tid < 4) sel[tid] = SNB - 1;
      __syncthreads();
      const unsigned long long Z = bin_hi[SNB - 1];
      d.tgt = d.nucleus ? (unsigned long long)((double)top_p * (double)Z) : Z;
      // the bin in which the cumulative mass first exceeds m
      auto bin_of = [&](unsigned long long m, int slot) {
        if (incl > m && incl - own <= m) sel[slot] = 2 * tid + (first <= m);
        __syncthreads();
        return sel[slot];
      };
      d.cut = d.nucleus ? bin_of(d.tgt, 0) : SNB;
      const unsigned long long lo = d.nucleus ? (d.cut > 0 ? bin_hi[d.cut - 1] : 0ull) : Z, hi = d.nucleus ? bin_hi[d.cut] : Z;
      d.cut_above = lo;
      d.p0 = bin_of(pick_mass(u, lo), 1);
      d.p1 = bin_of(pick_mass(u, hi), 2);
      d.pick_above = d.p0 > 0 ? bin_hi[d.p0 - 1] : 0ull;
      // this part's elements of those bins
      unsigned* count = (unsigned*)&sel[3];
      __syncthreads();
      if (tid == 0) *count = 0;
      __syncthreads();
      for_part(lg, part_at(V, g, np), part_at(V, g + 1, np), [&](float4 q, int at) {
        const float v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int bin = mass_bin(v[j], mx, d.scale);
          if ((bin >= d.p0 && bin <= d.p1) || bin == d.cut) {
            const unsigned i = atomicAdd(count, 1u);
            if (i < SCAP) sh.buf[i] = ((unsigned long long)order_key(v[j]) << 32) | (0xffffffffu - (uint32_t)(at + j));
          }
        }
      });
      __syncthreads();
      const unsigned mine = *count;
      if (tid == 0) base_sh = __hip_atomic_fetch_add(&w->listed, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      for (unsigned i = tid; i < min(mine, (unsigned)SCAP) && base_sh + i < SCAP; i += ST)
        __hip_atomic_store(&w->list[base_sh + i], sh.buf[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // this wave's write-through stores have left
      __syncthreads();
      if (tid == 0) base_sh = __hip_atomic_fetch_add(&w->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (base_sh != (unsigned)(np - 1)) return;
      const unsigned n = __hip_atomic_load(&w->listed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (n > SCAP) token = draw_row<1>(lg, V, mx, inv_t, top_p, u, h.best, sh_d);
      else if (n <= ST) token = pick_listed<1>(w, (int)n, d, sh.buf, scan, &sel[0]);
      else if (n <= 2 * ST) token = pick_listed<2>(w, (int)n, d, sh.buf, scan, &sel[0]);
      else token = pick_listed<SCAP / ST>(w, (int)n, d, sh.buf, scan, &sel[0]);
      if (token < 0 || token >= V) token = h.best;
    }
  }
  if (token < 0 || token >= V) token = 0;        // (a row without a single comparable logit: sample_kernel)
  if (tid == 0) {
    c.tokens_out[b] = token;
    if (c.logprob_out) c.logprob_out[b] = (c.forced && forced < 0) ? 0.f : (lg[token] - mx) * lp_scale - lp_lse;
    if (c.row_stats) { c.row_stats[2 * b] = mx; c.row_stats[2 * b + 1] = h.lse; }
    if (c.prob_row0_out) c.prob_row0_out[b] = __expf(c.logits[token] - row_head(ws, np).lse);     // softmax(logits)[0, token] (utils.py:363, row-0 quirk Q6)
  }
}

// probs = softmax(logits)[0, tokens] (utils.py:363, row-0 quirk Q6)
__global__ void prob_row0_kernel(const float* logits, const float* row_stats, const int32_t* tokens, float* out, int B) {
  const int b = threadIdx.x;
  if (b < B) out[b] = __expf(logits[tokens[b]] - row_stats[1]);
}

__global__ void advance_offsets_kernel(int32_t* offsets, const int32_t* rows, int B, int L) {
  const int i = threadIdx.x;
  if (i < B) offsets[rows ? rows[i] : i] += L;
}

__global__ void rope_tables_kernel(float* cos_tab, float* sin_tab, int max_pos, int D2, double base, double scale) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= max_pos * D2) return;
  const int pos = idx / D2, i = idx % D2;
  const double inv = pow(base, -2.0 * (double)i / (double)(2 * D2));
  const double ang = (double)pos * scale * inv;
  cos_tab[idx] = (float)cos(ang);
  sin_tab[idx] = (float)sin(ang);
}

template <typename S, typename T>
__global__ void convert_kernel(const S* src, T* dst, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) dst[i] = (T)(float)src[i];
}

}  // namespace

int launch_embed(const LinearW& W, const EmbedCall& c, hipStream_t st) {
  switch (c.act) {
    case MI_F32: return launch_embed_wk<float>(W, c, st);
    case MI_BF16: return launch_embed_wk<bf16>(W, c, st);
    case MI_F16: return launch_embed_wk<f16>(W, c, st);
  }
  return fail(MI_ERR_INVALID, "embed: bad activation dtype");
}

// rows' words, then the bins of their parts: no more parts than SAMPLE_WGS or one a row
static_assert(sizeof(SampleRow) % 16 == 0, "the bins are read 16 bytes at a time");
size_t sample_ws_bytes(int B) {
  const size_t rows = std::min(B, SAMPLE_SPLIT_ROWS);
  return rows * sizeof(SampleRow) + std::max<size_t>(SAMPLE_WGS, rows) * SNB * sizeof(unsigned long long);
}

static bool sample_draws(const SampleCall& c) { return c.forced == nullptr && (c.row_temp != nullptr || c.temperature != 0.f); }
bool sample_splits(const SampleCall& c) {
  const bool draws = sample_draws(c);
  return c.V >= (draws || c.top_logprobs > 0 ? SAMPLE_SPLIT_VOCAB : SAMPLE_SPLIT_GREEDY) &&
         c.B <= (!draws ? SAMPLE_SPLIT_ROWS_GREEDY : c.V < SAMPLE_SPLIT_WIDE ? SAMPLE_SPLIT_ROWS_NARROW : SAMPLE_SPLIT_ROWS) && row_vec(c.logits, c.V);
}

int launch_sample(const SampleCall& c, hipStream_t st) {
  if (c.B < 1) return fail(MI_ERR_INVALID, "sample: no rows");
  if (c.top_logprobs < 0 || c.top_logprobs > MI_MAX_TOP_LOGPROBS) return fail(MI_ERR_INVALID, "sample: top_logprobs out of range");
  if (c.ws != nullptr && sample_splits(c)) {
    const bool draws = sample_draws(c);
    SampleRow* ws = (SampleRow*)c.ws;
    unsigned long long* hist = (unsigned long long*)(ws + c.B);
    const bool scaled = c.lp_temp && (c.row_temp != nullptr || (c.temperature > 0.f && c.temperature != 1.f));
    const int np = std::max(1, std::min(SG, SAMPLE_WGS / c.B - (c.top_logprobs > 0))), nwg = draws ? np : 1;
    hipLaunchKernelGGL(sample_parts_kernel, dim3(np, c.B), dim3(ST), 0, st, c, ws);
    MI_HIP(hipGetLastError());
    if (draws || scaled) hipLaunchKernelGGL(sample_masses_kernel, dim3(np, c.B), dim3(ST), 0, st, c, ws, hist);
    MI_HIP(hipGetLastError());
    hipLaunchKernelGGL(sample_draw_kernel, dim3(nwg + (c.top_logprobs > 0), c.B), dim3(ST), 0, st, c, ws, hist, np, nwg);
    MI_HIP(hipGetLastError());
    return MI_OK;
  }
  hipLaunchKernelGGL(sample_kernel, dim3(c.B), dim3(ST), 0, st, c);
  MI_HIP(hipGetLastError());
  if (c.prob_row0_out) {
    hipLaunchKernelGGL(prob_row0_kernel, dim3(1), dim3(64 * ((c.B + 63) / 64)), 0, st, c.logits, c.row_stats,
                       c.tokens_out, c.prob_row0_out, c.B);
    MI_HIP(hipGetLastError());
  }
  return MI_OK;
}

__global__ __launch_bounds__(256) void gather_rows_kernel(const u128* src, size_t row_vecs, const int32_t* idx, u128* dst) {
  const u128* s = src + (size_t)idx[blockIdx.x] * row_vecs;
  u128* d = dst + (size_t)blockIdx.x * row_vecs;
  for (size_t i = threadIdx.x; i < row_vecs; i += 256) d[i] = s[i];
}

int launch_gather_rows(const void* src, size_t row_bytes, const int32_t* idx, int n, void* dst, hipStream_t st) {
  if (row_bytes % 16 != 0) return fail(MI_ERR_UNSUPPORTED, "gather_rows: rows must be multiples of 16 bytes");
  if (n <= 0) return MI_OK;
  hipLaunchKernelGGL(gather_rows_kernel, dim3(n), dim3(256), 0, st, (const u128*)src, row_bytes / 16, idx, (u128*)dst);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_advance_offsets(int32_t* offsets, const int32_t* rows, int B, int L, hipStream_t st) {
  hipLaunchKernelGGL(advance_offsets_kernel, dim3(1), dim3(64 * ((B + 63) / 64)), 0, st, offsets, rows, B, L);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_rope_tables(float* cos_tab, float* sin_tab, int max_pos, int D, float base, float scale, hipStream_t st) {
  const int n = max_pos * (D / 2);
  hipLaunchKernelGGL(rope_tables_kernel, dim3((n + 255) / 256), dim3(256), 0, st, cos_tab, sin_tab, max_pos, D / 2,
                     (double)base, (double)scale);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_convert(const void* src, int sdt, void* dst, int ddt, size_t n, hipStream_t st) {
  const dim3 grid((unsigned)std::min<size_t>((n + 255) / 256, 4096)), block(256);
#define CV(S, T) hipLaunchKernelGGL((convert_kernel<S, T>), grid, block, 0, st, (const S*)src, (T*)dst, n)
  if (sdt == MI_F32 && ddt == MI_F32) CV(float, float);
  else if (sdt == MI_BF16 && ddt == MI_F32) CV(bf16, float);
  else if (sdt == MI_F16 && ddt == MI_F32) CV(f16, float);
  else if (sdt == MI_F32 && ddt == MI_BF16) CV(float, bf16);
  else if (sdt == MI_F32 && ddt == MI_F16) CV(float, f16);
  else if (sdt == MI_BF16 && ddt == MI_BF16) CV(bf16, bf16);
  else if (sdt == MI_F16 && ddt == MI_F16) CV(f16, f16);
  else return fail(MI_ERR_UNSUPPORTED, "convert: dtype pair not supported");
#undef CV
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
