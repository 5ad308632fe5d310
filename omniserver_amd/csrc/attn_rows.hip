// Packed prefill / append attention on 32-row tiles (the decoder's 128-wide heads).
#include "attn_rows.h"

// ---------------------------------------------------------------------------
// The tile structure and what bounds it are in attn_rows.h.  One 4096-token prompt, 12
// heads / 2 KV heads, MI355X: 69 us = 745 TFLOP/s, where 16-row tiles of 16 x 16 x 32 MFMAs
// took 193 us; of the 69 about 45 are arithmetic, the rest the tiles' staging and the
// causal tail.  Staging through registers instead of straight to LDS: 82 us.  Two wave groups
// kept half a step apart (one in its MFMAs while the other is in its softmax): 74 us.
// ---------------------------------------------------------------------------
#define AR_HD 128

struct RowsArgs {
  const half_t* q;
  int q_stride;
  const half_t* k_cache;
  const half_t* v_cache;
  int pool_rows, max_len, nkv, G;
  const int64_t* slots;    // [T]
  const int64_t* kv_len;   // [T]
  const int* qblocks;      // [nqb][2] = (first token, count)
  half_t* out;
  int out_stride;
  float scale_log2;
};

// A workgroup takes one query block (n <= 32 R / G consecutive tokens of one segment) and
// one KV head: its n G rows, token-major, in R tiles of 32, so that every K / V byte staged
// in LDS serves all query heads of the group and a tile's rows end within a few keys of
// each other.  The block's key tiles are dealt to S groups of R waves (group s takes a
// contiguous run), each with its own LDS tiles, and the S states of a row meet in LDS at
// the end: S shortens the longest block's chain, R sets how many rows share a staged tile.
// Tile rows are 256 bytes: K with its 16-byte chunks XOR-swizzled by row % 16, V with its
// 64-byte quarters XOR-swizzled by row % 4, which makes the operand reads conflict-free.
// With R = 1 a group is one wave, which needs no barrier and no second buffer.
template <int R, int S, int KT>
__global__ __launch_bounds__(64 * R * S, 2) void attn_rows_kernel(RowsArgs a) {
  constexpr int NBUF = R == 1 ? 1 : 2;
  constexpr int TB = KT * AR_HD * 2;                // bytes of a K (or V) tile
  constexpr int NL = TB / 1024;                     // 1 KB (4-row) pieces of a tile
  constexpr int NB = KT / 32;
  constexpr int MB = R * S * 64 * 64 * 4;           // the merge's outputs
  constexpr int SB = S * NBUF * 2 * TB > MB ? S * NBUF * 2 * TB : MB;
  __shared__ __attribute__((aligned(16))) char smem[SB];
  __shared__ float ml_lds[S][R][2][32];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / R;                          // key group
  const int rt = wave - grp * R;                     // row tile
  const int l32 = lane & 31, h = lane >> 5;
  const int item = (int)gridDim.x - 1 - (int)blockIdx.x;   // a segment's last blocks first
  const int qb = item / a.nkv;
  const int g = item - qb * a.nkv;
  const int t0 = a.qblocks[2 * qb];
  const int n = min(a.qblocks[2 * qb + 1], 32 * R / a.G);
  const int64_t slot = a.slots[t0];
  if (slot < 0 || slot >= a.pool_rows || n <= 0) return;   // the whole workgroup
  const int nrows = n * a.G;
  const int row = min(32 * rt + l32, nrows - 1);
  const int tok = t0 + row / a.G;
  const int u = row - (row / a.G) * a.G;
  const int64_t lim64 = a.kv_len[tok];
  const int lim = (int)(lim64 < 1 ? 1 : lim64 > a.max_len ? a.max_len : lim64);
  const int lim_lo = __builtin_amdgcn_readfirstlane(lim);                 // rows ascend
  const int lim_hi = __builtin_amdgcn_readlane(lim, 31);
  const int64_t end64 = a.kv_len[t0 + n - 1];
  const int end = (int)(end64 < 1 ? 1 : end64 > a.max_len ? a.max_len : end64);
  const bool rows_here = 32 * rt < nrows;

  half8_t qf[8];
  {
    const half_t* qp = a.q + (int64_t)tok * a.q_stride + (int64_t)(g * a.G + u) * AR_HD + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = *(const half8_t*)(qp + 16 * ks);
  }

  const int ntiles = (end + KT - 1) / KT;
  const int steps = (ntiles + S - 1) / S;
  const int tbeg = grp * steps;
  const int nt = min(steps, ntiles - tbeg);          // may be <= 0

  // R = 1 stages through registers (its one buffer is free only once the tile is used): chunk
  // c = lane + 64 j of a tile is row c / 16, 16-byte chunk c % 16.
  const int cr = lane >> 4, cc = lane & 15;
  const int64_t tstride = (int64_t)a.nkv * AR_HD;    // halfs per token
  const int64_t base = slot * (int64_t)a.max_len * tstride + g * AR_HD;
  const half_t* kb0 = a.k_cache + base;
  const half_t* vb0 = a.v_cache + base;
  const uint32_t coff = (uint32_t)((int64_t)cr * tstride + cc * 8) * 2;
  half8_t kr[NL], vr[NL];
  auto load_tile = [&](int tb) {
    if (tb + KT <= end) {            // uniform bases, one lane offset for every chunk
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int64_t off = (int64_t)(tb + 4 * j) * tstride;
        kr[j] = *(const half8_t*)((const char*)(kb0 + off) + coff);
        vr[j] = *(const half8_t*)((const char*)(vb0 + off) + coff);
      }
    } else {                         // the last tile repeats the block's last key
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int t = min(tb + cr + 4 * j, end - 1);
        const int64_t off = (int64_t)t * tstride + cc * 8;
        kr[j] = *(const half8_t*)(kb0 + off);
        vr[j] = *(const half8_t*)(vb0 + off);
      }
    }
  };
  auto store_tile = [&](char* kt) {
    char* vt = kt + TB;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int r = cr + 4 * j;
      *(half8_t*)(kt + r * 256 + ((cc ^ (r & 15)) << 4)) = kr[j];
      *(half8_t*)(vt + r * 256 + ((cc << 4) ^ ((r & 3) << 6))) = vr[j];
    }
  };

  float m_run = -INFINITY, l_run = 0.f;
  f32x16 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;

  // K fragment (key 32 b + l32, dims 16 ks + 8 h ..) at kt + 8192 b + (koff ^ 32 ks);
  // V fragment (dims 32 d + 16 (lane / 16 % 2) + .., keys 16 t + 4 h .. and + 8) at
  // vt + 4096 t (+ 2048) + (voff ^ 64 d)
  const int koff = l32 * 256 + ((h ^ (l32 & 15)) << 4);
  const int i16 = lane & 15;
  const int voff = (4 * h + (i16 >> 2)) * 256 + ((i16 >> 2) << 6) + ((lane >> 4) & 1) * 32 +
                   (i16 & 3) * 8;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  f32x16 s[NB];
  half8_t p[2 * NB];
  auto scores = [&](const char* kt) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[b][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        s[b] = mfma32x32x16(*(const half8_t*)(kt + 8192 * b + (koff ^ (ks << 5))), qf[ks], s[b]);
    // the first reads ahead, then one step's reads beside each step's MFMAs
    __builtin_amdgcn_sched_group_barrier(0x100, 3 * NB, 0);
#pragma unroll
    for (int ks = 0; ks < 5; ++ks) {
      __builtin_amdgcn_sched_group_barrier(0x008, NB, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, NB, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 3 * NB, 0);
  };
  auto mask = [&](int tb) {
    if (tb + KT > lim_lo) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (tb + 32 * b + 8 * (i >> 2) + 4 * h + (i & 3) >= lim) s[b][i] = -INFINITY;
    }
  };
  auto output = [&](const char* vt) {
#pragma unroll
    for (int t = 0; t < 2 * NB; ++t)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const char* vp = vt + 4096 * t + (voff ^ (d << 6));
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)vp);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vp + 2048));
        const half4_t a0 = __builtin_bit_cast(half4_t, lo), a1 = __builtin_bit_cast(half4_t, hi);
        o[d] = mfma32x32x16((half8_t){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]},
                            p[t], o[d]);
      }
  };

  char* gbuf = smem + grp * NBUF * 2 * TB;
  // R > 1 stages straight to LDS, 1 KB per instruction, the swizzle in the source addresses.
  auto dma_half = [&](int tb, char* dst, const half_t* src0, bool is_k) {
    const uint32_t l0 = __builtin_amdgcn_readfirstlane(lds_offset(dst)) + rt * 1024;
    const bool whole = tb + KT <= end;               // else the block's last key is repeated
    const half_t* src = src0 + (int64_t)tb * tstride;
#pragma unroll
    for (int j = 0; j < NL / R; ++j) {
      const int r0 = 4 * (rt + R * j), r = r0 + cr;
      const int ch = is_k ? cc ^ (r & 15) : cc ^ ((r & 3) << 2);
      const half_t* sp = whole ? src + (int64_t)r0 * tstride : src;
      const int rr = whole ? cr : min(r, end - 1 - tb);
      dma16(sp, (uint32_t)rr * (uint32_t)tstride * 2 + ch * 16, l0 + R * j * 1024);
    }
  };
  auto dma_tile = [&](int tb, char* kt) {
    dma_half(tb, kt, kb0, true);
    dma_half(tb, kt + TB, vb0, false);
  };
  if (nt > 0) {
    if constexpr (R > 1) dma_tile(tbeg * KT, gbuf);
    else load_tile(tbeg * KT);
  }
  // Q has landed: without this the compiler counts the Q loads as outstanding inside the loop
  // and makes every tile's first MFMAs wait for the transfers just requested
  __builtin_amdgcn_s_waitcnt(0x0f70);
  for (int it = 0; it < steps; ++it) {
    char* kt = gbuf + (NBUF == 2 ? (it & 1) * 2 * TB : 0);
    const int tb = (tbeg + it) * KT;
    if constexpr (R > 1) {
      vm_wait();             // this wave's part of tile it has landed; so, past the barrier,
      lds_barrier();         // have the others', and tile it - 1's buffer is free
      if (it + 1 < nt) dma_tile(tb + KT, gbuf + ((it + 1) & 1) * 2 * TB);
    } else {
      if (it < nt) store_tile(kt);
      if (it + 1 < nt) load_tile(tb + KT);
    }
    if (it < nt && rows_here && tb < lim_hi) {
      scores(kt);
      mask(tb);
      softmax32<NB, 4>(s, a.scale_log2, m_run, l_run, o, p);
      output(kt + TB);
    }
  }

  // Every group's unnormalised output and (max, sum) per row go to LDS; wave (rt, grp)
  // merges its share of the 16 output quads (4 dims) of row tile rt over the S groups.
  {
    float x, y;
    half_pair(l_run, x, y);
    l_run = x + y;
  }
  __syncthreads();
  float* om = (float*)smem;
  if (rows_here) {
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        *(float4*)(om + (((grp * R + rt) * 16 + 4 * d + b) * 64 + lane) * 4) =
            make_float4(o[d][4 * b], o[d][4 * b + 1], o[d][4 * b + 2], o[d][4 * b + 3]);
    if (h == 0) {
      ml_lds[grp][rt][0][l32] = m_run;
      ml_lds[grp][rt][1][l32] = l_run;
    }
  }
  __syncthreads();
  if (!rows_here) return;
  float M = ml_lds[0][rt][0][l32];       // key 0 is in the first group: finite
#pragma unroll
  for (int s = 1; s < S; ++s) M = fmaxf(M, ml_lds[s][rt][0][l32]);
  float f[S], den = 0.f;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    f[s] = __builtin_amdgcn_exp2f(ml_lds[s][rt][0][l32] - M);    // -inf: a group without keys
    den += ml_lds[s][rt][1][l32] * f[s];
  }
  const float inv = 1.0f / den;
  half_t* op = a.out + (int64_t)tok * a.out_stride + (int64_t)(g * a.G + u) * AR_HD;
  constexpr int NQ = 16 / S;
#pragma unroll
  for (int k = 0; k < NQ; k += 2) {
    unsigned w[2][2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int quad = grp * NQ + k + e;
      float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const float4 v = *(const float4*)(om + (((s * R + rt) * 16 + quad) * 64 + lane) * 4);
        acc.x = fmaf(v.x, f[s], acc.x);
        acc.y = fmaf(v.y, f[s], acc.y);
        acc.z = fmaf(v.z, f[s], acc.z);
        acc.w = fmaf(v.w, f[s], acc.w);
      }
      const half2_t c0 = {(half_t)(acc.x * inv), (half_t)(acc.y * inv)};
      const half2_t c1 = {(half_t)(acc.z * inv), (half_t)(acc.w * inv)};
      w[e][0] = __builtin_bit_cast(unsigned, c0);
      w[e][1] = __builtin_bit_cast(unsigned, c1);
    }
    // lane half h holds dims 8 quad + 4 h .. + 3 of quads k and k + 1: exchanged, half 0 has
    // all 8 dims of quad k and half 1 those of quad k + 1
    const auto r0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
    const auto r1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
    const u32x4 st = {r0[0], r1[0], r0[1], r1[1]};
    if (32 * rt + l32 < nrows) *(u32x4*)(op + 8 * (grp * NQ + k + h)) = st;
  }
}

// Causal varlen attention of packed query tokens over their pool rows, as
// omni_prefill_attention, on 32-row tiles of (token, query head) pairs.  (rows, groups) of a
// workgroup: (128, 1), (128, 2), (64, 4) or (32, 8); qblocks counts are at most
// rows / (n_heads / n_kv_heads) tokens, which must be at least 1.
extern "C" int omni_prefill_attention_rows(const void* q, int q_stride, const void* k_cache,
                                           const void* v_cache, int pool_rows, int max_len,
                                           const int64_t* slots, const int64_t* kv_len,
                                           const int* qblocks, int nqb, void* out, int out_stride,
                                           int n_heads, int n_kv_heads, int head_dim, float scale,
                                           int rows, int groups, void* stream) {
  if (nqb < 0 || n_heads <= 0 || n_kv_heads <= 0 || pool_rows <= 0 || max_len <= 0) return OMNI_EINVAL;
  if (head_dim != AR_HD || n_heads % n_kv_heads) return OMNI_EUNSUPPORTED;
  const int form = rows == 128 && (groups == 1 || groups == 2) ? groups
                   : rows == 64 && groups == 4 ? 4 : rows == 32 && groups == 8 ? 8 : 0;
  if (!form) return OMNI_EINVAL;
  if (n_heads / n_kv_heads > rows || !(scale > 0.f)) return OMNI_EUNSUPPORTED;
  if (q_stride < n_heads * AR_HD || (q_stride & 7)) return OMNI_EINVAL;
  if (out_stride < n_heads * AR_HD || (out_stride & 7)) return OMNI_EINVAL;
  if (nqb == 0) return OMNI_OK;
  if (!q || !k_cache || !v_cache || !slots || !kv_len || !qblocks || !out) return OMNI_EINVAL;
  if (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15) return OMNI_EINVAL;
  const int64_t grid = (int64_t)nqb * n_kv_heads;
  if (grid > 0x7fffffff) return OMNI_EUNSUPPORTED;
  RowsArgs a;
  a.q = (const half_t*)q;
  a.q_stride = q_stride;
  a.k_cache = (const half_t*)k_cache;
  a.v_cache = (const half_t*)v_cache;
  a.pool_rows = pool_rows;
  a.max_len = max_len;
  a.nkv = n_kv_heads;
  a.G = n_heads / n_kv_heads;
  a.slots = slots;
  a.kv_len = kv_len;
  a.qblocks = qblocks;
  a.out = (half_t*)out;
  a.out_stride = out_stride;
  a.scale_log2 = scale * 1.4426950408889634f;
  const dim3 gd((unsigned)grid);
  hipStream_t st = (hipStream_t)stream;
  if (form == 1)
    hipLaunchKernelGGL((attn_rows_kernel<4, 1, 64>), gd, dim3(256), 0, st, a);
  else if (form == 2)
    hipLaunchKernelGGL((attn_rows_kernel<4, 2, 64>), gd, dim3(512), 0, st, a);
  else if (form == 4)
    hipLaunchKernelGGL((attn_rows_kernel<2, 4, 32>), gd, dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((attn_rows_kernel<1, 8, 32>), gd, dim3(512), 0, st, a);
  OMNI_CHECK_LAUNCH();
  return OMNI_OK;
}
