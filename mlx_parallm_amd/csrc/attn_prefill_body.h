// attn_prefill_body.h -- the causal attention of a query tile on 16-bit caches (attn_prefill.hip, and beside the decoding rows of a mixed step: attn_decode.hip)
#pragma once
#include <type_traits>

#include "kernels.h"

namespace mi {
namespace prefill {

constexpr int PREFILL_MAX_SLICES = 16;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <typename T>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (std::is_same<T, bf16>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ void pack2_split(float a, float b, uint32_t& hi, uint32_t& lo) {   // as in attn_decode.hip
  const T ha = (T)a, hb = (T)b;
  T h[2] = {ha, hb};
  T l[2] = {(T)(a - (float)ha), (T)(b - (float)hb)};
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, l);
}

template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  T v[2] = {(T)a, (T)b};
  return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ u32x4 load16_agent(const void* p) {       // (as in gemv_phase.h: past this XCD's L2)
  const unsigned long long* q = (const unsigned long long*)p;
  const unsigned long long a = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned long long b = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
}
__device__ __forceinline__ void store16_agent(void* p, const f32x4& v) {
  unsigned long long* q = (unsigned long long*)p;
  __hip_atomic_store(q, ((unsigned long long)__float_as_uint(v.y) << 32) | __float_as_uint(v.x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(q + 1, ((unsigned long long)__float_as_uint(v.w) << 32) | __float_as_uint(v.z), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Keys split over gridDim.z workgroups: a chunk of a prompt that enters next to decoding sequences has few query tiles (32 tokens x 8
// kv heads: 16 workgroups for 256 CUs) and walked all its keys in one chain of dependent blocks -- 58 us at 640 keys (Qwen3-14B
// heads, rocprof) whatever the chip could do.  A row has its own number of slices nz <= gridDim.z (prefill_row_slices), so what a row
// gets depends on the call's shape and its own keys, not on how many its neighbours have cached.
// Slice z takes key blocks [z nb / nz, (z + 1) nb / nz), leaves (m, l, O) and counts itself;
// the last one of a tile adds the slices in order (no spinning; hand-off as in gemm_skinny.hip).  l: summed over the lanes of a query.
// false: not the last.  part: [tile][slice][wave][64 lanes][DT + 1] x 16 bytes.
template <int DT>
__device__ __forceinline__ bool join_slices(const AttnCall& c, int tile, int nz, int zi, int nzi, int* last_sh, int waves, int wave, int lane, f32x4 (&acc)[DT], float& m, float& l) {
  float* base = c.partial + ((size_t)tile * nzi * waves + wave) * (64 * (DT + 1) * 4) + lane * 4;
  const size_t slice = (size_t)waves * (64 * (DT + 1) * 4);
  float* mine = base + zi * slice;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) store16_agent(mine + dt * 256, acc[dt]);
  store16_agent(mine + DT * 256, f32x4{m, l, 0.f, 0.f});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    int* cp = c.counters + tile;
    const int old = __hip_atomic_fetch_add(cp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == nz - 1) __hip_atomic_store(cp, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);       // for the next launch
    *last_sh = old == nz - 1;
  }
  __syncthreads();
  if (!*last_sh) return false;
  float mz[PREFILL_MAX_SLICES], lz[PREFILL_MAX_SLICES];
  m = -1e30f;
#pragma unroll
  for (int i = 0; i < PREFILL_MAX_SLICES; ++i) {
    // (m, l) alone: with the unused half of the 16 bytes in the same registers hipcc waited for every slice's before the next went out
    const unsigned long long v = __hip_atomic_load((const unsigned long long*)(base + (size_t)min(i, nz - 1) * slice + DT * 256),
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    mz[i] = i < nz ? __uint_as_float((uint32_t)v) : -INFINITY;
    lz[i] = __uint_as_float((uint32_t)(v >> 32));
  }
#pragma unroll
  for (int i = 0; i < PREFILL_MAX_SLICES; ++i) m = fmaxf(m, mz[i]);
  l = 0.f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i0 = 0; i0 < PREFILL_MAX_SLICES; i0 += 2) {
    if (i0 >= nz) break;                              // (uniform)
    u32x4 v[2][DT];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) v[j][dt] = load16_agent(base + (size_t)min(i0 + j, nz - 1) * slice + dt * 256);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float w = __builtin_amdgcn_exp2f(mz[i0 + j] - m);          // (a slice past the last: exp2(-inf) = 0)
      l += lz[i0 + j] * w;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[dt][r] += __uint_as_float(v[j][dt][r]) * w;
    }
  }
  return true;
}

constexpr int QT = 16;      // queries per query group (one MFMA column set)
constexpr int KB = 32;      // keys per block

// one KiB: global (per-lane source address) -> LDS at a wave-uniform address (lane-linear)
__device__ __forceinline__ void dma_kib(const void* gsrc, unsigned lds_dst) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(gsrc), "s"(lds_dst) : "memory");
}

template <int D> constexpr size_t attn_prefill_dma_lds() { return 6 * (size_t)KB * D * 2 + 16; }      // three K and V images, the join's flag

// qt, bh, zi of (tiles, .., nzi): the workgroup's query tile, (row, kv head) and slice; only its first G waves come here
template <typename T, int D, int G, bool PAGED, int QG, bool SPLIT>
__device__ __forceinline__ void attn_prefill_dma_body(const AttnCall& c, const int qt, const int bh, const int tiles, const int zi, const int nzi, unsigned char* smem) {
  static_assert(sizeof(T) == 2 && D % 32 == 0 && D <= 128, "16-bit activations / caches, head_dim 32..128");
  constexpr int KK = D / 32, DT = D / 16, NT = G * 64;
  constexpr int QTT = QT * QG;                        // queries per workgroup
  constexpr int NPIECE = KB * D / 8;                  // 16-byte pieces of one K (or V) block
  constexpr int NP = (NPIECE + NT - 1) / NT;          // per thread
  constexpr int IMG = KB * D * 2;                     // bytes of one image
  constexpr float LOG2E = 1.4426950408889634f;
  const AttnShape& s = c.s;
  const int b = bh / s.Hkv, kh = bh % s.Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g4 = lane >> 4;
  const int kb = s.rows ? s.rows[b] : b;              // cache row of batch entry b
  const int off = c.offsets[kb];
  const int t0 = qt * QTT;
  const int nk = off + min(t0 + QTT, s.L);            // keys any query of the tile may see
  const int nb = (nk + KB - 1) / KB;
  // this slice's blocks.  A workgroup beyond its row's slices has none and leaves at the end (a return here instead: 22.6 us against 22.2 at a chunk
  // of 32 tokens behind 700 keys, Qwen3-14B heads)
  const int nz = SPLIT ? prefill_row_slices(nzi, off + s.L, c.join_cost, c.slice_cost) : 1, z = SPLIT ? min(zi, nz) : 0;
  const int j0 = SPLIT ? z * nb / nz : 0, j1 = SPLIT ? min(z + 1, nz) * nb / nz : nb;
  const int h = kh * G + wave;

  // K / V blocks go global -> LDS by LDS-DMA into a ring of THREE buffers: block j + 2 is issued at the head of
  // iteration j (into the buffer block j - 1 was read from: every wave finished those reads before the barrier that
  // closed iteration j - 1) and waited for at the end of iteration j + 1 (s_waitcnt vmcnt(that block's DMAs of this
  // wave), then the barrier: the block is everybody's).  No staging registers, no ds_write -- and no compiler-visible
  // vector loads in the loop: with K / V loaded into registers hipcc's wait-count pass put s_waitcnt vmcnt(0) at the head
  // of the loop body (a register-reuse hazard it could not rule out across the back edge), which drained the prefetch
  // just issued and exposed a memory round trip every block: 268 us per layer at 8 x 1024 tokens against 191 here.
  // The images are those of attn_prefill_kernel; a DMA writes lane-linear, so the layout is realised through each
  // lane's SOURCE address: K instruction i covers slots 64 i .. 64 i + 63 of [16-key tile][kk][g][key & 15], V
  // instruction i the 32 keys x 32 bytes of 16-d tile i.
  constexpr int NINST = NPIECE / 64;                  // DMA instructions per image and block
  constexpr int CNT = (NINST + G - 1) / G;            // per wave (the last wave may repeat the last instruction: same bytes, same place)
  unsigned char (*kimg)[IMG] = (unsigned char (*)[IMG])smem;
  unsigned char (*vimg)[IMG] = kimg + 3;
  const unsigned k_lds = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem, v_lds = k_lds + 3 * IMG;

  const T* kc = (const T*)c.kcache;
  const T* vc = (const T*)c.vcache;
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  auto dma_block = [&](int j, int buf) {
#pragma unroll
    for (int n = 0; n < CNT; ++n) {
      const int i = min(wv + G * n, NINST - 1);
      {   // K: slot S = 64 i + lane = (((kt * KK + kk) * 4 + dclo) * 16 + klo)
        const int S = i * 64 + lane;
        const int klo = S & 15, dclo = (S >> 4) & 3, tk = S >> 6, kk = tk % KK, kt = tk / KK;
        const int key = min(j * KB + kt * 16 + klo, nk - 1);
        const T* src = kc + kv_elem<PAGED>(s, kb, kh, key) + 8 * (kk * 4 + dclo);
        dma_kib(src, k_lds + buf * IMG + i * 1024);
      }
      {   // V: slot S = dt * 64 + key * 2 + (dc & 1)
        const int key = min(j * KB + (lane >> 1), nk - 1);
        const T* src = vc + kv_elem<PAGED>(s, kb, kh, key) + 8 * (i * 2 + (lane & 1));
        dma_kib(src, v_lds + buf * IMG + i * 1024);
      }
    }
  };

  // Q^T fragments of this wave's head (B operand: column = query), one set per query group
  u32x4 qf[QG][KK];
  int tq[QG];
#pragma unroll
  for (int u = 0; u < QG; ++u) {
    tq[u] = min(t0 + QT * u + c16, s.L - 1);          // this lane's query of group u (clamped; stores are guarded)
    const T* qp = (const T*)c.q + ((size_t)b * s.L + tq[u]) * s.Hq * D + (size_t)h * D;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[u][kk] = *(const u32x4*)(qp + 32 * kk + 8 * g4);
  }
  dma_block(j0, 0);
  dma_block(j0 + 1, 1);                               // (past the last block: clamped keys, masked)
  // the Q fragments count as loaded from here on (hipcc waits for its own loads with vmcnt(0): blocks 0 and 1 have landed too)
#pragma unroll
  for (int u = 0; u < QG; ++u)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) asm volatile("" :: "v"(qf[u][kk]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const float sc2 = c.scale * LOG2E;
  float m_run[QG], l_run[QG];
  f32x4 accO[QG][DT];
#pragma unroll
  for (int u = 0; u < QG; ++u) {
    m_run[u] = -1e30f; l_run[u] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) accO[u][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int tq4 = c16 >> 2, tp = c16 & 3;

  int buf = 0;                                        // (j - j0) mod 3
  for (int j = j0; j < j1; ++j) {
    const int bnext2 = buf == 0 ? 2 : buf - 1;        // (j - j0 + 2) mod 3
    dma_block(j + 2, bnext2);
    f32x4 sc[QG][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int u = 0; u < QG; ++u) sc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const u32x4 kf = *(const u32x4*)(kimg[buf] + (((t * KK + kk) * 4 + g4) * 16 + c16) * 16);
#pragma unroll
        for (int u = 0; u < QG; ++u) sc[u][t] = mfma16<T>(kf, qf[u][kk], sc[u][t]);
      }
    }
    u32x4 pf[QG], pl[QG];                             // P = hi + lo, two 16-bit operands (attn_decode.hip pack2_split)
#pragma unroll
    for (int u = 0; u < QG; ++u) {
      // The vector ALU, not the matrix core, bounds this loop (~110 vector instructions + 9 transcendentals per 16 MFMAs
      // as first written), so: the causal mask only in the blocks that reach past the group's first query (uniform), the
      // scale folded into the exponent's FMA, and O / l rescaled only when some query's running max moved (uniform;
      // multiplying by exp2(0) = 1 is the identity, so skipping it changes no bit).
      const int qpos = off + t0 + QT * u + c16;       // key positions <= qpos are visible to this lane's query of group u
      float mx = -INFINITY;
      if (j * KB + KB - 1 > off + t0 + QT * u) {      // a diagonal block of this group
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool ok = (j * KB + 16 * t + 4 * g4 + r) <= qpos;
            sc[u][t][r] = ok ? sc[u][t][r] : -INFINITY;
          }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[u][t][r]);
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m_run[u], mx * sc2);     // (scale > 0: the largest raw score is the largest scaled one)
      if (__builtin_amdgcn_ballot_w64(mn != m_run[u]) != 0) {
        const float corr = __builtin_amdgcn_exp2f(m_run[u] - mn);
        m_run[u] = mn;
        l_run[u] *= corr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) accO[u][dt] *= corr;
      }
      float p[2][4];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) { p[t][r] = __builtin_amdgcn_exp2f(fmaf(sc[u][t][r], sc2, -mn)); l_run[u] += p[t][r]; }
      uint32_t ph[4], pw[4];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        pack2_split<T>(p[t][0], p[t][1], ph[2 * t], pw[2 * t]);
        pack2_split<T>(p[t][2], p[t][3], ph[2 * t + 1], pw[2 * t + 1]);
      }
      pf[u] = u32x4{ph[0], ph[1], ph[2], ph[3]};
      pl[u] = u32x4{pw[0], pw[1], pw[2], pw[3]};
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const unsigned char* a0 = vimg[buf] + (size_t)dt * (KB * 32) + (4 * g4 + tq4) * 32 + tp * 8;
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)a0);
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(a0 + 16 * 32));
      const uint32_t* w0 = (const uint32_t*)&v0;
      const uint32_t* w1 = (const uint32_t*)&v1;
      const u32x4 vf = {w0[0], w0[1], w1[0], w1[1]};
#pragma unroll
      for (int u = 0; u < QG; ++u) {
        accO[u][dt] = mfma16<T>(vf, pf[u], accO[u][dt]);
        accO[u][dt] = mfma16<T>(vf, pl[u], accO[u][dt]);
      }
    }
    // lgkmcnt(0): every LDS read of this iteration has RETURNED before the barrier lets another wave issue the DMA that
    // overwrites this buffer's predecessor -- hipcc may sink an MFMA, and the wait in front of it, below the barrier, and
    // under load (four workgroups per CU on the LDS queue) a read issued just before the barrier was still queued when a
    // fast wave's DMA landed: wrong tiles that came and went with the load on the chip (tests/test_gpu_fullsize.py).
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "i"(2 * CNT) : "memory");    // and block j + 1 has landed (block j + 2 may still fly)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    buf = buf == 2 ? 0 : buf + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // no DMA of this workgroup may land after it has left the CU
  if (SPLIT && z == nz) return;

#pragma unroll
  for (int u = 0; u < QG; ++u) {
    float l = l_run[u];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if constexpr (SPLIT) {                            // (launched with one query group only)
      if (nz > 1 && !join_slices<DT>(c, bh * tiles + qt, nz, zi, nzi, (int*)(smem + 6 * IMG), G, wave, lane, accO[u], m_run[u], l)) return;
    }
    if (t0 + QT * u + c16 < s.L) {
      const float inv = 1.0f / l;
      if (c.frag_mt > 0) {                            // (uniform) 8 k of the output linear's x from a pair of lanes: elements j and j + 4 of them share a word
        const int row = c.frag_row0 + b * s.L + tq[u];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const u32x2 v = {pack2<T>(accO[u][dt][0] * inv, accO[u][dt][1] * inv), pack2<T>(accO[u][dt][2] * inv, accO[u][dt][3] * inv)};
          const u32x2 w = {(uint32_t)__shfl_xor((int)v.x, 16, 64), (uint32_t)__shfl_xor((int)v.y, 16, 64)};
          if ((g4 & 1) == 0)
            *(u32x4*)((T*)c.out + q4_frag_elem(row, h * D + 16 * dt + 4 * g4, c.frag_mt, s.Hq * D / 64)) =
                u32x4{(v.x & 0xffffu) | w.x << 16, v.x >> 16 | (w.x & 0xffff0000u), (v.y & 0xffffu) | w.y << 16, v.y >> 16 | (w.y & 0xffff0000u)};
        }
        continue;
      }
      T* op = (T*)c.out + ((size_t)b * s.L + tq[u]) * s.Hq * D + (size_t)h * D + 4 * g4;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const u32x2 v = {pack2<T>(accO[u][dt][0] * inv, accO[u][dt][1] * inv), pack2<T>(accO[u][dt][2] * inv, accO[u][dt][3] * inv)};
        *(u32x2*)(op + 16 * dt) = v;
      }
    }
  }
}

}  // namespace prefill
}  // namespace mi
