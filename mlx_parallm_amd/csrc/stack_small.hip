// stack_small.hip -- a decode step or a prompt of a small model, all layers in ONE launch (float32 activations: float32 models, and the float32-cache mode).
//
// A model of some 10^4 weights a layer has nothing to stream: its step is the launches, six a layer of 3 to 5 us each (64 wide, eight layers, 4-bit:
// 200 us a token).  A row needs no other row, so one workgroup walks all layers of its row: every matrix is spread over the 512 threads, in registers, and a thread
// asks for its words of the NEXT layer as soon as this layer's are used; the cached keys and values, which do not depend on the layer, come at its start.  What is
// left is a chain of five barriers a layer and the instructions between them (one CU's): 43 us that step, the whole token 250 -> 76.  On the way, us: 14
// barriers, a thread per number 72; five, and sizes of the split known at run time alone 61; no division in the loop 51; the split fixed 43.
// The same arithmetic as the kernels it replaces: weights as scale * code + bias with two roundings, products and sums in float32, layer 0 up to its attention
// rounded to the model's type (`rnd0`).  Prompts: small_prompt_kernel.  The limits (64 wide, 256 outputs of q|k|v and of gate|up, 128 columns of o and down) are
// those at which a layer's float32 weights fill the threads' registers (222 to 240 of 256); codes take 84, and no model of codes alone that is wider has been tried.  256 keys because a
// row's keys are one workgroup's: longer ones take the launches, whose attention splits them.
#include <type_traits>

#include "kernels.h"

namespace mi {

namespace {

constexpr int NT = 512;
// The threads' share of a matrix: q|k|v and gate|up ("big") 256 columns x 2 groups of at most 32 k, o and down 64 x 8 of 16.  PER: k values of a word
template <bool BIG> struct Split { static constexpr int COLS = BIG ? 256 : 64, GROUPS = NT / COLS, KS = BIG ? 32 : 16; };
template <int KIND> struct Kind { static constexpr int PER = KIND == SMALL_F32 ? 1 : KIND == SMALL_CODES ? 4 : 2; };

// a thread's part of a matrix: column n, words [w0, w0 + cnt) of it, the first `cut` of them in one quantisation group
struct Part { int n, w0, cnt, cut; };
__device__ __forceinline__ Part part_of(bool big, int N, int words, int group, int tid, int g) {      // g = tid / columns
  const int groups = big ? Split<true>::GROUPS : Split<false>::GROUPS;
  Part p;
  p.n = min(tid - g * (NT / groups), N - 1);
  p.w0 = g * words / groups;
  p.cnt = (g + 1) * words / groups - p.w0;
  p.cut = (p.w0 * 4 / group + 1) * group / 4 - p.w0;
  return p;
}
template <bool BIG>
__device__ __forceinline__ Part part_of(int N, int words, int group) {                                // (g is the same in a wave)
  return part_of(BIG, N, words, group, threadIdx.x, __builtin_amdgcn_readfirstlane(threadIdx.x / Split<BIG>::COLS));
}

// ---- packing: a matrix as [MW][NT] words, the i-th of every thread, and (codes) [2][NT] scales | biases, of the groups of its first and last -----------
__device__ __forceinline__ uint32_t code_at(const LinearW& W, size_t row, int k, int bits) {
  if (bits == 4) {
    const uint32_t v = W.layout ? *(const uint32_t*)((const char*)W.w + tiled_block_q4(row, k, W.K) + tiled_q4_code_off(row, k & ~7))
                                : ((const uint32_t*)W.w)[row * (W.K / 8) + k / 8];
    return (v >> (4 * (k & 7))) & 15u;
  }
  return W.layout ? *((const uint8_t*)W.w + tiled_block_q8(row, k, W.K) + tiled_q8_code_off(row, k)) : ((const uint8_t*)W.w)[row * W.K + k];
}
template <typename T>
__device__ __forceinline__ float2 scale_at(const LinearW& W, size_t row, int k, int bits) {
  if (W.layout) {
    const char* b = (const char*)W.w + (bits == 4 ? tiled_block_q4(row, k, W.K) + tiled_q4_scale_off(row, k) : tiled_block_q8(row, k, W.K) + tiled_q8_scale_off(row));
    return float2{(float)*(const T*)b, (float)*(const T*)(b + (bits == 4 ? 64 : 32))};
  }
  const size_t i = row * (W.K / W.group) + k / W.group;
  return float2{(float)((const T*)W.scales)[i], (float)((const T*)W.biases)[i]};
}
__global__ __launch_bounds__(NT) void small_pack_kernel(LinearW W, bool big, int kind, int bits, int sdt, uint32_t* words, float2* sb) {
  const int per = kind == SMALL_F32 ? 1 : kind == SMALL_CODES ? 4 : 2, tid = threadIdx.x, i = blockIdx.x;
  const Part p = part_of(big, W.N, W.K / per, W.group, tid, tid / (big ? Split<true>::COLS : Split<false>::COLS));
  const int last = max(p.cnt - 1, 0), n = p.n, k = (p.w0 + min(i, last)) * per;          // (past the last: that one again)
  uint32_t v = 0;
  if (kind == SMALL_F32) v = ((const uint32_t*)W.w)[(size_t)n * W.K + k];
  else if (kind == SMALL_CODES) for (int j = 0; j < 4; ++j) v |= code_at(W, n, k + j, bits) << (8 * j);
  else for (int j = 0; j < 2; ++j)
    v |= (uint32_t)*(W.layout ? (const uint16_t*)((const char*)W.w + tiled_piece_dense16(n, (k + j) & ~7, W.K)) + ((k + j) & 7) : (const uint16_t*)W.w + (size_t)n * W.K + k + j) << (16 * j);
  words[i * NT + tid] = v;
  if (kind == SMALL_CODES && i < 2) {
    const int at = (p.w0 + i * last) * per;
    sb[i * NT + tid] = sdt == MI_F32 ? scale_at<float>(W, n, at, bits) : sdt == MI_BF16 ? scale_at<bf16>(W, n, at, bits) : scale_at<f16>(W, n, at, bits);
  }
}

template <int KIND, bool BIG>
struct Regs {
  static constexpr int PER = Kind<KIND>::PER, MW = Split<BIG>::KS / PER, WORDS = MW * NT;
  static constexpr bool CODES = KIND == SMALL_CODES;
  uint32_t w[MW];
  float2 sb[CODES ? 2 : 1];                           // (groups of 32 and more: two of them)
  __device__ __forceinline__ void load(const uint32_t* words, const float2* scales) {
#pragma unroll
    for (int i = 0; i < MW; ++i) w[i] = words[i * NT + threadIdx.x];
    if constexpr (CODES) { sb[0] = scales[threadIdx.x]; sb[1] = scales[NT + threadIdx.x]; }
  }
  __device__ __forceinline__ float dot(const Part& p, const float* x) const {
    float acc[2] = {0.f, 0.f};
    int cnt = p.cnt, cut = p.cut;
    asm volatile("" : "+s"(cnt), "+s"(cut));          // (compared here, not kept as a mask per word over all layers)
    const float* xk = x + p.w0 * PER;
#pragma unroll
    for (int i = 0; i < MW; ++i) {
      if (i < cnt) {                                  // (uniform; a break keeps longer loops rolled, the words in scratch)
      float& a = acc[i & 1];
      if constexpr (KIND == SMALL_F32) a = fmaf(__uint_as_float(w[i]), xk[i], a);
      else if constexpr (KIND == SMALL_BF16) a = fmaf(bf16hi(w[i]), xk[2 * i + 1], fmaf(bf16lo(w[i]), xk[2 * i], a));
      else if constexpr (KIND == SMALL_F16) {
        const f16* h = (const f16*)&w[i];
        a = fmaf((float)h[1], xk[2 * i + 1], fmaf((float)h[0], xk[2 * i], a));
      } else {
        const float sx = i < cut ? sb[0].x : sb[1].x, sy = i < cut ? sb[0].y : sb[1].y;
        const float4 xv = *(const float4*)(xk + 4 * i);
        a = fmaf(mul_add_unfused((float)(w[i] & 255u), sx, sy), xv.x, a);
        a = fmaf(mul_add_unfused((float)((w[i] >> 8) & 255u), sx, sy), xv.y, a);
        a = fmaf(mul_add_unfused((float)((w[i] >> 16) & 255u), sx, sy), xv.z, a);
        a = fmaf(mul_add_unfused((float)(w[i] >> 24), sx, sy), xv.w, a);
      }
      }
    }
    return acc[0] + acc[1];
  }
  // The same for n rows x[t][LD], eight or four a time: a weight is multiplied out once for all of them.  Rows behind the n-th are read (the arrays have PT of
  // them) and their sums dropped: a condition per row and word costs more.  out: [n][NT]
  template <int M, int LD>
  __device__ __forceinline__ void some(const Part& p, const float* x, int m, float* out) const {
    float acc[M];
    int cnt = p.cnt, cut = p.cut;
    asm volatile("" : "+s"(cnt), "+s"(cut));
    const float* xk = x + p.w0 * PER;
#pragma unroll
    for (int t = 0; t < M; ++t) acc[t] = 0.f;
#pragma unroll
    for (int i = 0; i < MW; ++i) {
      if (i < cnt) {
        float v[PER];
        if constexpr (KIND == SMALL_F32) v[0] = __uint_as_float(w[i]);
        else if constexpr (KIND == SMALL_BF16) { v[0] = bf16lo(w[i]); v[1] = bf16hi(w[i]); }
        else if constexpr (KIND == SMALL_F16) { const f16* h = (const f16*)&w[i]; v[0] = (float)h[0]; v[1] = (float)h[1]; }
        else {
          const float sx = i < cut ? sb[0].x : sb[1].x, sy = i < cut ? sb[0].y : sb[1].y;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = mul_add_unfused((float)((w[i] >> (8 * j)) & 255u), sx, sy);
        }
#pragma unroll
        for (int t = 0; t < M; ++t) {
          const float* xt = xk + t * LD + PER * i;
          if constexpr (PER == 4) {
            const float4 q = *(const float4*)xt;
            acc[t] = fmaf(v[3], q.w, fmaf(v[2], q.z, fmaf(v[1], q.y, fmaf(v[0], q.x, acc[t]))));
          } else {
#pragma unroll
            for (int j = 0; j < PER; ++j) acc[t] = fmaf(v[j], xt[j], acc[t]);
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < M; ++t)
      if (t < m) out[t * NT + threadIdx.x] = acc[t];
  }
  template <int LD>
  __device__ __forceinline__ void dots(const Part& p, const float* x, int n, float* out) const {
    for (int t = 0; t < n; t += 8) {
      if (n - t > 4) some<8, LD>(p, x + t * LD, n - t, out + t * NT);
      else some<4, LD>(p, x + t * LD, n - t, out + t * NT);
    }
  }
};
// the groups' sums of column n, in their order
template <bool BIG>
__device__ __forceinline__ float join(const float* part, int n) {
  float t[Split<BIG>::GROUPS], v = 0.f;
#pragma unroll
  for (int g = 0; g < Split<BIG>::GROUPS; ++g) t[g] = part[g * Split<BIG>::COLS + n];
#pragma unroll
  for (int g = 0; g < Split<BIG>::GROUPS; ++g) v += t[g];
  return v;
}
// what a wave has written to LDS is there for its own reads (its operations complete in order)
__device__ __forceinline__ void wave_lds() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// what the workgroup has written to LDS is there; loads stay in flight (__syncthreads would wait for the next layer's words at every barrier)
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// What needs the sums of a matrix -- residual, norm, rotation, gated unit -- every wave makes for the whole row, the same numbers at the same places of LDS: a barrier
// stands only between a matrix's partial sums (two buffers in turn) and what joins them, and behind the heads.  A wave has whole heads: keys over its lanes.
template <int KIND, int D, bool PAGED>
__global__ __launch_bounds__(NT) void stack_small_kernel(SmallStackCall c) {
  constexpr bool AHEAD = KIND != SMALL_F32 || D == 16;           // a layer's cached keys and values asked for at its start (float32 words leave no registers for heads of 32)
  constexpr int PER = Kind<KIND>::PER, NW = NT / 64, NV = AHEAD ? 8 : 0, KG = 64 / D;
  constexpr float LOG2E = 1.4426950408889634f;
  __shared__ __attribute__((aligned(16))) float xn[64], p0[NT], p1[NT], qk[256], vn[128], ov[128], act[128];
  __shared__ float sc[NW][SMALL_MAX_KEYS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), b = blockIdx.x;
  const int H = c.H, Hq = c.s.Hq, Hkv = c.s.Hkv, G = Hq / Hkv, nq = Hq * D, nkv = Hkv * D, I = c.I;
  const int kb = c.s.rows ? c.s.rows[b] : b, pos = c.offsets[kb];
  const Part pq = part_of<true>(nq + 2 * nkv, H / PER, c.group), po = part_of<false>(H, nq / PER, c.group), pg = part_of<true>(2 * I, H / PER, c.group), pd = part_of<false>(H, I / PER, c.group);
  Regs<KIND, true> rq, rg;
  Regs<KIND, false> ro, rd;
  constexpr int OW = rq.WORDS, GW = OW + ro.WORDS, DW = GW + rg.WORDS, LW = DW + rd.WORDS;      // words of a layer: q|k|v, o, gate|up, down
  rq.load(c.words, c.scales);
  ro.load(c.words + OW, c.scales + 2 * NT);
  rg.load(c.words + GW, c.scales + 4 * NT);
  rd.load(c.words + DW, c.scales + 6 * NT);
  const int col = min(lane, H - 1);
  float x = lane < H ? c.x[(size_t)b * H + lane] : 0.f;         // a lane per column of the row
  const int ri = lane % (D / 2);                      // a lane's rotation: the same for every 64 / (D / 2) heads
  const float cs = c.cos_tab[(size_t)pos * (D / 2) + ri], sn = c.sin_tab[(size_t)pos * (D / 2) + ri];
  const float sc2 = c.scale * LOG2E;
  const int h0 = min(wave, Hq - 1) / G;

  float n1 = c.norms[col], n2 = c.norms[H + col];     // the two norms' weights
  auto norm = [&](float nw, int rnd) {                // -> xn
    const float rs = 1.0f / sqrtf(wave_sum(x * x) / (float)H + c.eps);
    float v = x * rs;
    if (rnd != RND_NONE) v = round_rt(round_rt(v, rnd) * nw, rnd);
    else v *= nw;
    xn[lane] = v;
    wave_lds();
  };
  for (int l = 0; l < c.layers; ++l) {
    const int rnd = l == 0 ? c.rnd0 : RND_NONE;
    const int nl = min(l + 1, c.layers - 1);
    const uint32_t* wn = c.words + (size_t)nl * LW;
    const float2* sbn = c.scales + (size_t)nl * 8 * NT;
    float* kc = c.kcache + (size_t)l * c.layer_elems;
    float* vc = c.vcache + (size_t)l * c.layer_elems;
    // cached keys and values of this wave's first head: key `lane`, value column lane % D of keys lane / D + KG i
    const int last = max(pos - 1, 0);
    float4 kr[D / 4];
    float vr[NV + 1];
    if constexpr (AHEAD) {
      const float4* src = (const float4*)(kc + kv_elem<PAGED>(c.s, kb, h0, min(lane, last)));
#pragma unroll
      for (int e = 0; e < D / 4; ++e) kr[e] = src[e];
#pragma unroll
      for (int i = 0; i < NV; ++i) vr[i] = vc[kv_elem<PAGED>(c.s, kb, h0, min(lane / D + KG * i, last)) + lane % D];
    }
    norm(n1, rnd);
    n1 = c.norms[2 * nl * H + col];
    p0[tid] = rq.dot(pq, xn);
    rq.load(wn, sbn);
    lds_barrier();
    // q, k: rotated pairs (i, i + D / 2) of a head; v as it is
    for (int t = lane; t < (Hq + Hkv) * (D / 2); t += 64) {
      const int n = t / (D / 2) * D + ri;             // (k's heads stand behind q's)
      float a = join<true>(p0, n), e = join<true>(p0, n + D / 2);
      if (rnd != RND_NONE) { a = round_rt(a, rnd); e = round_rt(e, rnd); }
      float ra = a * cs - e * sn, re = a * sn + e * cs;
      if (rnd != RND_NONE) { ra = round_rt(ra, rnd); re = round_rt(re, rnd); }
      qk[n] = ra; qk[n + D / 2] = re;
      if (wave == 0 && n >= nq) {
        float* dst = kc + kv_elem<PAGED>(c.s, kb, (n - nq) / D, pos) + ri;
        dst[0] = ra; dst[D / 2] = re;
      }
    }
    for (int t = lane; t < nkv; t += 64) {
      const float v = round_rt(join<true>(p0, nq + nkv + t), rnd);
      vn[t] = v;
      if (wave == 0) vc[kv_elem<PAGED>(c.s, kb, t / D, pos) + t % D] = v;
    }
    wave_lds();
    for (int h = wave; h < Hq; h += NW) {
      const int hk = h == wave ? h0 : h / G;
      const float* q = qk + h * D;
      float* s = sc[wave];
      float mx = -1e30f;
      auto dot_key = [&](const float4 (&k)[D / 4]) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < D / 4; ++e) d = fmaf(k[e].w, q[4 * e + 3], fmaf(k[e].z, q[4 * e + 2], fmaf(k[e].y, q[4 * e + 1], fmaf(k[e].x, q[4 * e], d))));
        return d;
      };
      for (int j = lane; j <= pos; j += 64) {
        float d;
        if (AHEAD && h == wave && j < 64) d = dot_key(kr);       // (uniform: h and the trip)
        else {
          float4 k[D / 4];
          const float4* src = (const float4*)(kc + kv_elem<PAGED>(c.s, kb, hk, min(j, last)));
#pragma unroll
          for (int e = 0; e < D / 4; ++e) k[e] = src[e];
          d = dot_key(k);
        }
        if (j == pos) {
          float4 k[D / 4];
#pragma unroll
          for (int e = 0; e < D / 4; ++e) k[e] = *(const float4*)(qk + nq + hk * D + 4 * e);
          d = dot_key(k);
        }
        s[j] = d * sc2;
        mx = fmaxf(mx, s[j]);
      }
      mx = wave_max(mx);
      float t = 0.f;
      for (int j = lane; j <= pos; j += 64) { const float e = __builtin_amdgcn_exp2f(s[j] - mx); s[j] = e; t += e; }
      t = wave_sum(t);
      wave_lds();
      float o = 0.f;
      const float v1 = vn[hk * D + lane % D];
      if (AHEAD && h == wave) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const int j = lane / D + KG * i;
          if (j <= pos) o = fmaf(s[j], j < pos ? vr[i] : v1, o);
        }
      }
      for (int j = lane / D + (h == wave ? KG * NV : 0); j <= pos; j += KG)
        o = fmaf(s[j], j < pos ? vc[kv_elem<PAGED>(c.s, kb, hk, j) + lane % D] : v1, o);
#pragma unroll
      for (int m = D; m < 64; m <<= 1) o += __shfl_xor(o, m, 64);
      if (lane < D) ov[h * D + lane] = o / t;
      wave_lds();                                     // (s is written again for the next head)
    }
    lds_barrier();
    p1[tid] = ro.dot(po, ov);
    ro.load(wn + OW, sbn + 2 * NT);
    lds_barrier();
    if (lane < H) x += join<false>(p1, lane);
    norm(n2, RND_NONE);
    n2 = c.norms[(2 * nl + 1) * H + col];
    p0[tid] = rg.dot(pg, xn);
    rg.load(wn + GW, sbn + 4 * NT);
    lds_barrier();
#pragma unroll
    for (int k = lane; k < 128; k += 64) {
      if (k < I) {
        const float g = join<true>(p0, k), u = join<true>(p0, I + k);
        act[k] = g * (1.0f / (1.0f + expf(-g))) * u;
      }
    }
    wave_lds();
    p1[tid] = rd.dot(pd, act);
    rd.load(wn + DW, sbn + 6 * NT);
    lds_barrier();
    if (lane < H) x += join<false>(p1, lane);
  }
  if (wave == 0) {
    if (lane < H) c.h[(size_t)b * H + lane] = x;
    if (lane == 0) c.offsets[kb] = pos + 1;           // (nobody else reads it in this step)
  }
}

// The prompt of a small model, all layers in one launch: a workgroup a row again, PT tokens a time through all layers (their keys and values are the next ones' cache).
// A wave owns every NW-th token (its columns over the lanes, residual, norm, rotation, gated unit) and takes whole (token, head)s of the attention; the matrices are
// multiplied by all threads, PT rows a time.  Nine tokens of two rows, eight layers, 4-bit, with the logits: 643 us -> 196, 32 rows of them 7.3 -> 0.6 ms.
constexpr int PT = 16;
constexpr size_t prompt_lds() { return (size_t)(PT * (64 + 2 * NT + 256 + 2 * 128) + NT / 64 * SMALL_MAX_KEYS) * 4; }
template <int KIND, int D, bool PAGED>
__global__ __launch_bounds__(NT) void small_prompt_kernel(SmallStackCall c) {
  constexpr int PER = Kind<KIND>::PER, NW = NT / 64, KG = 64 / D, OWN = PT / NW;
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* xn = lds;                                    // [PT][64]
  float* p0 = xn + PT * 64;                           // [PT][NT]
  float* p1 = p0 + PT * NT;                           // [PT][NT]
  float* qkv = p1 + PT * NT;                          // [PT][256]
  float* ov = qkv + PT * 256;                         // [PT][128]
  float* act = ov + PT * 128;                         // [PT][128]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), b = blockIdx.x;
  float* s = act + PT * 128 + wave * SMALL_MAX_KEYS;  // [SMALL_MAX_KEYS]: this wave's scores
  const int H = c.H, Hq = c.s.Hq, Hkv = c.s.Hkv, G = Hq / Hkv, nq = Hq * D, nkv = Hkv * D, I = c.I, L = c.s.L;
  const int kb = c.s.rows ? c.s.rows[b] : b, before = c.offsets[kb];
  if (c.upto < SMALL_MAX_KEYS && before > c.upto) return;       // (uniform)
  const Part pq = part_of<true>(nq + 2 * nkv, H / PER, c.group), po = part_of<false>(H, nq / PER, c.group), pg = part_of<true>(2 * I, H / PER, c.group), pd = part_of<false>(H, I / PER, c.group);
  Regs<KIND, true> rq, rg;
  Regs<KIND, false> ro, rd;
  constexpr int OW = rq.WORDS, GW = OW + ro.WORDS, DW = GW + rg.WORDS, LW = DW + rd.WORDS;
  rq.load(c.words, c.scales);
  ro.load(c.words + OW, c.scales + 2 * NT);
  rg.load(c.words + GW, c.scales + 4 * NT);
  rd.load(c.words + DW, c.scales + 6 * NT);
  const int col = min(lane, H - 1), ri = lane % (D / 2);
  const float sc2 = c.scale * LOG2E;
  float n1 = c.norms[col], n2 = c.norms[H + col];
  for (int t0 = 0; t0 < L; t0 += PT) {
    const int n = min(PT, L - t0), pos = before + t0; // pos: cached keys in front of these tokens
    float x[OWN], cs[OWN], sn[OWN];
#pragma unroll
    for (int u = 0; u < OWN; ++u) {
      const int t = min(wave + NW * u, n - 1);
      x[u] = c.x[((size_t)b * L + t0 + t) * H + col];
      if (lane >= H) x[u] = 0.f;
      cs[u] = c.cos_tab[(size_t)(pos + t) * (D / 2) + ri]; sn[u] = c.sin_tab[(size_t)(pos + t) * (D / 2) + ri];
    }
    auto norm = [&](float nw, int rnd) {
#pragma unroll
      for (int u = 0; u < OWN; ++u) {
        const int t = wave + NW * u;
        if (t >= n) break;                            // (uniform)
        const float rs = 1.0f / sqrtf(wave_sum(x[u] * x[u]) / (float)H + c.eps);
        float v = x[u] * rs;
        if (rnd != RND_NONE) v = round_rt(round_rt(v, rnd) * nw, rnd);
        else v *= nw;
        xn[t * 64 + lane] = v;
      }
    };
    for (int l = 0; l < c.layers; ++l) {
      const int rnd = l == 0 ? c.rnd0 : RND_NONE;
      const int nl = l + 1 < c.layers ? l + 1 : 0;    // (behind the last one: the first again, for the next tokens)
      const uint32_t* wn = c.words + (size_t)nl * LW;
      const float2* sbn = c.scales + (size_t)nl * 8 * NT;
      float* kc = c.kcache + (size_t)l * c.layer_elems;
      float* vc = c.vcache + (size_t)l * c.layer_elems;
      norm(n1, rnd);
      n1 = c.norms[2 * nl * H + col];
      lds_barrier();
      rq.template dots<64>(pq, xn, n, p0);
      rq.load(wn, sbn);
      lds_barrier();
#pragma unroll
      for (int u = 0; u < OWN; ++u) {
        const int t = wave + NW * u;
        if (t >= n) break;
        const float* p = p0 + t * NT;
        float* row = qkv + t * 256;
        for (int e = lane; e < (Hq + Hkv) * (D / 2); e += 64) {
          const int i = e / (D / 2) * D + ri;
          float a = join<true>(p, i), v = join<true>(p, i + D / 2);
          if (rnd != RND_NONE) { a = round_rt(a, rnd); v = round_rt(v, rnd); }
          float ra = a * cs[u] - v * sn[u], rv = a * sn[u] + v * cs[u];
          if (rnd != RND_NONE) { ra = round_rt(ra, rnd); rv = round_rt(rv, rnd); }
          row[i] = ra; row[i + D / 2] = rv;
          if (i >= nq) {
            float* dst = kc + kv_elem<PAGED>(c.s, kb, (i - nq) / D, pos + t) + ri;
            dst[0] = ra; dst[D / 2] = rv;
          }
        }
        for (int e = lane; e < nkv; e += 64) {
          const float v = round_rt(join<true>(p, nq + nkv + e), rnd);
          row[nq + nkv + e] = v;
          vc[kv_elem<PAGED>(c.s, kb, e / D, pos + t) + e % D] = v;
        }
      }
      lds_barrier();
      for (int pr = wave; pr < n * Hq; pr += NW) {    // token t, head h: the cached keys, then those of tokens 0 .. t
        const int t = pr / Hq, h = pr - t * Hq, hk = h / G;
        const float* q = qkv + t * 256 + h * D;
        float mx = -1e30f;
        auto score = [&](const float* k, int j) {
          float d = 0.f;
#pragma unroll
          for (int e = 0; e < D / 4; ++e) {
            const float4 a = *(const float4*)(k + 4 * e), w = *(const float4*)(q + 4 * e);
            d = fmaf(a.w, w.w, fmaf(a.z, w.z, fmaf(a.y, w.y, fmaf(a.x, w.x, d))));
          }
          s[j] = d * sc2;
          mx = fmaxf(mx, d * sc2);
        };
        for (int j = lane; j < pos; j += 64) score(kc + kv_elem<PAGED>(c.s, kb, hk, j), j);
        if (lane <= t) score(qkv + lane * 256 + nq + hk * D, pos + lane);
        mx = wave_max(mx);
        wave_lds();
        float sum = 0.f;
        for (int j = lane; j <= pos + t; j += 64) { const float e = __builtin_amdgcn_exp2f(s[j] - mx); s[j] = e; sum += e; }
        sum = wave_sum(sum);
        wave_lds();
        float o = 0.f;
        for (int j = lane / D; j < pos; j += KG) o = fmaf(s[j], vc[kv_elem<PAGED>(c.s, kb, hk, j) + lane % D], o);
        for (int j = lane / D; j <= t; j += KG) o = fmaf(s[pos + j], qkv[j * 256 + nq + nkv + hk * D + lane % D], o);
#pragma unroll
        for (int m = D; m < 64; m <<= 1) o += __shfl_xor(o, m, 64);
        if (lane < D) ov[t * 128 + h * D + lane] = o / sum;
        wave_lds();                                   // (s is written again)
      }
      lds_barrier();
      ro.template dots<128>(po, ov, n, p1);
      ro.load(wn + OW, sbn + 2 * NT);
      lds_barrier();
      auto add = [&]() {
#pragma unroll
        for (int u = 0; u < OWN; ++u)
          if (wave + NW * u < n && lane < H) x[u] += join<false>(p1 + (wave + NW * u) * NT, lane);
      };
      add();
      norm(n2, RND_NONE);
      n2 = c.norms[(2 * nl + 1) * H + col];
      lds_barrier();
      rg.template dots<64>(pg, xn, n, p0);
      rg.load(wn + GW, sbn + 4 * NT);
      lds_barrier();
#pragma unroll
      for (int u = 0; u < OWN; ++u) {
        const int t = wave + NW * u;
        if (t >= n) break;
        for (int k = lane; k < I; k += 64) {
          const float g = join<true>(p0 + t * NT, k), up = join<true>(p0 + t * NT, I + k);
          act[t * 128 + k] = g * (1.0f / (1.0f + expf(-g))) * up;
        }
      }
      lds_barrier();
      rd.template dots<128>(pd, act, n, p1);
      rd.load(wn + DW, sbn + 6 * NT);
      lds_barrier();
      add();
    }
#pragma unroll
    for (int u = 0; u < OWN; ++u)
      if (wave + NW * u < n && lane < H) c.h[((size_t)b * L + t0 + wave + NW * u) * H + lane] = x[u];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // these keys and values are the next tokens' cache
    __syncthreads();
  }
  if (tid == 0 && c.advance) c.offsets[kb] = before + L;           // (read at the head, in front of many barriers)
}

int per_of(int kind) { return kind == SMALL_F32 ? 1 : kind == SMALL_CODES ? 4 : 2; }
int kind_of(const LinearW& W) { return wk_is_quant(W.wk) ? SMALL_CODES : W.wk == WK_F32 ? SMALL_F32 : W.wk == WK_BF16 ? SMALL_BF16 : SMALL_F16; }

}  // namespace

// does a matrix fit the threads' registers?  (Adapters are the launches': the kernels have no second product, and one may be set before the weights are complete)
bool small_stack_fits(const LinearW& W, bool big) {
  if (W.lora_b[0] != nullptr || W.lora_b[1] != nullptr) return false;
  const int kind = kind_of(W), per = per_of(kind);
  return W.N <= (big ? 256 : 64) && W.K <= (big ? 64 : 128) && W.K % per == 0 && (kind != SMALL_CODES || (W.group % 32 == 0 && W.K % W.group == 0));
}
int small_stack_kind(const LinearW& W) { return kind_of(W); }
size_t small_stack_words(int kind, bool big) { return (size_t)NT * (big ? 32 : 16) / per_of(kind); }
size_t small_stack_scales(int kind) { return kind == SMALL_CODES ? 2 * NT : 0; }
bool small_stack_shape(int H, int heads, int kv_heads, int D, int I) {
  return H <= 64 && I <= 128 && heads * D <= 128 && (D == 16 || D == 32) && heads % kv_heads == 0;
}

int launch_small_pack(const LinearW& W, bool big, uint32_t* words, float2* sb, hipStream_t st) {
  const int kind = kind_of(W), mw = (int)(small_stack_words(kind, big) / NT);
  hipLaunchKernelGGL(small_pack_kernel, dim3(mw), dim3(NT), 0, st, W, big, kind, wk_bits(W.wk), wk_is_quant(W.wk) ? wk_scale_dtype(W.wk) : 0, words, sb);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_stack_small(const SmallStackCall& c, hipStream_t st) {
  if (!small_stack_shape(c.H, c.s.Hq, c.s.Hkv, c.s.D, c.I) || c.s.act != MI_F32 || c.s.kv != MI_F32 || c.s.L < 1) return fail(MI_ERR_UNSUPPORTED, "stack_small: shape / dtype not supported");
#define GOP(K, DV, PG) do { auto kern = small_prompt_kernel<K, DV, PG>; \
    static std::atomic<bool> granted[64]; \
    MI_TRY(grant_lds((const void*)kern, prompt_lds(), granted)); \
    hipLaunchKernelGGL(kern, dim3(c.s.B), dim3(NT), prompt_lds(), st, c); } while (0)
#define GO(K, DV) do { if (c.s.L > 1) { if (c.s.btab) GOP(K, DV, true); else GOP(K, DV, false); } \
    else if (c.s.btab) hipLaunchKernelGGL((stack_small_kernel<K, DV, true>), dim3(c.s.B), dim3(NT), 0, st, c); \
    else hipLaunchKernelGGL((stack_small_kernel<K, DV, false>), dim3(c.s.B), dim3(NT), 0, st, c); } while (0)
#define GOK(K) do { if (c.s.D == 16) GO(K, 16); else GO(K, 32); } while (0)
  switch (c.kind) {
    case SMALL_F32: GOK(SMALL_F32); break;
    case SMALL_BF16: GOK(SMALL_BF16); break;
    case SMALL_F16: GOK(SMALL_F16); break;
    case SMALL_CODES: GOK(SMALL_CODES); break;
    default: return fail(MI_ERR_INVALID, "stack_small: bad kind");
  }
#undef GOK
#undef GO
#undef GOP
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
