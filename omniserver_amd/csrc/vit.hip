// Vision tower (Qwen2-VL ViT) kernels: LayerNorm (also over a split-K linear's partial
// sums, with its bias and residual add), the 2-D vision rotary, and non-causal segmented
// attention at head_dim 80.  The tower's linears run on the pipelined fp16 GEMM over packed
// weights (gemm_pipe.hip, omni_f16_gemm_pipe_packed: bias / QuickGELU / GELU / residual /
// partial-sum epilogues) and the patch embedding on the tiled one (gemv.hip).
//
// Replaces, per block of model/qwen2_vit.py:36-69: nn.LayerNorm (norm1 / norm2, and
// the merger's ln_q at :128), the fused rotary of kernels/vision_rope.py:19-47, and
// the varlen flash call at :58-63 (cu_seqlens separate the images; every patch of an
// image attends to every patch of the same image).
#include "attn_rows.h"

// ---------------------------------------------------------------------------
// LayerNorm over rows: y = (x - mean) * rsqrt(var + eps) * w + b, fp32 math, fp16 out
// (biased variance, as nn.LayerNorm).  One wave per row; lane holds 16-byte chunks
// lane + 64 u (u < 4), so N <= 2048.
// ---------------------------------------------------------------------------
#define LN_MAXCH 4

// PARTS: x is formed first, as a split-K linear's finish with the residual epilogue would
// form it (gemm_pipe_finish_kernel, GP_RESID): h = fp16(sum of the nparts fp32 slices
// [nparts][M][N] in slice order (+ bias, before the rounding)), x = fp16(res + h), with the
// residual rows read from x (row stride ldx) and x written to x_out (which may alias them:
// each lane reads its chunks before it writes them).
template <bool PARTS>
__global__ __launch_bounds__(256) void layernorm_kernel(const half_t* x, int ldx,
                                                        const half_t* __restrict__ w,
                                                        const half_t* __restrict__ b, int M,
                                                        int N, float eps, half_t* out, int ldo,
                                                        const float* __restrict__ parts = nullptr,
                                                        int nparts = 0,
                                                        const half_t* __restrict__ pbias = nullptr,
                                                        half_t* x_out = nullptr, int ldxo = 0) {
#pragma clang fp contract(off)
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const int lane = threadIdx.x & 63;
  const int nc = N >> 3;
  const half_t* xr = x + (int64_t)row * ldx;
  float v[LN_MAXCH][8];
  float s = 0.f;
#pragma unroll
  for (int u = 0; u < LN_MAXCH; ++u) {
    const int c = lane + 64 * u;
    half8_t h = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};
    if (c < nc) {
      h = *(const half8_t*)(xr + c * 8);
      if (PARTS) {
        const float* pp = parts + (int64_t)row * N + c * 8;
        const int64_t ps = (int64_t)M * N;
        float a[8];
        const float4 lo = *(const float4*)pp, hi = *(const float4*)(pp + 4);
        a[0] = lo.x; a[1] = lo.y; a[2] = lo.z; a[3] = lo.w;
        a[4] = hi.x; a[5] = hi.y; a[6] = hi.z; a[7] = hi.w;
        for (int p = 1; p < nparts; ++p) {
          const float4 l2 = *(const float4*)(pp + p * ps), h2 = *(const float4*)(pp + p * ps + 4);
          a[0] += l2.x; a[1] += l2.y; a[2] += l2.z; a[3] += l2.w;
          a[4] += h2.x; a[5] += h2.y; a[6] += h2.z; a[7] += h2.w;
        }
        half8_t bb = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};
        if (pbias) bb = *(const half8_t*)(pbias + c * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const half_t lin = pbias ? (half_t)(a[e] + (float)bb[e]) : (half_t)a[e];
          h[e] = (half_t)((float)h[e] + (float)lin);
        }
        *(half8_t*)(x_out + (int64_t)row * ldxo + c * 8) = h;
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[u][e] = (float)h[e];
      s += v[u][e];
    }
  }
  const float mean = wave_sum(s) / (float)N;
  float q = 0.f;
#pragma unroll
  for (int u = 0; u < LN_MAXCH; ++u) {
    if (lane + 64 * u < nc) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = v[u][e] - mean;
        q += d * d;
      }
    }
  }
  const float var = wave_sum(q) / (float)N;
  const float rstd = rsqrtf(var + eps);
#pragma unroll
  for (int u = 0; u < LN_MAXCH; ++u) {
    const int c = lane + 64 * u;
    if (c >= nc) continue;
    const half8_t wv = *(const half8_t*)(w + c * 8);
    const half8_t bv = *(const half8_t*)(b + c * 8);
    half8_t y;
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (half_t)((v[u][e] - mean) * rstd * (float)wv[e] + (float)bv[e]);
    *(half8_t*)(out + (int64_t)row * ldo + c * 8) = y;
  }
}

// Rows of N = 256 NC (the tower's 1280: NC = 5): lane l holds the 4-column chunks
// l + 64 u, u < NC, so every lane has the same work and every load of the row - the
// residual / input, NP fp32 partial slices, the linear's bias and the norm's gains - goes out
// before any arithmetic (the kernel above waits chunk by chunk, and its 8-column chunks give
// lanes 2 or 3 of them at N = 1280).  NP = 0: plain LayerNorm of x; NP > 0: x formed first
// from the slices as in the kernel above.  Sums in this kernel's own order (chunks u, then
// the 4 columns), so its outputs agree with the kernel above to fp32 rounding of the mean
// and variance, and its two forms with each other bit for bit.
template <int NC, int NP>
__global__ __launch_bounds__(256) void layernorm4_kernel(const half_t* x, int ldx,
                                                         const half_t* __restrict__ w,
                                                         const half_t* __restrict__ b, int M,
                                                         float eps, half_t* out, int ldo,
                                                         const float* __restrict__ parts,
                                                         const half_t* __restrict__ pbias,
                                                         half_t* x_out, int ldxo) {
#pragma clang fp contract(off)
  constexpr int N = 256 * NC;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const int lane = threadIdx.x & 63;
  const half_t* xr = x + (int64_t)row * ldx + 4 * lane;
  half4_t xv[NC], wv[NC], bv[NC], pb[NP > 0 ? NC : 1];
  float4 pv[NP > 0 ? NP : 1][NC];
#pragma unroll
  for (int u = 0; u < NC; ++u) {
    xv[u] = *(const half4_t*)(xr + 256 * u);
    if (NP > 0) {
#pragma unroll
      for (int p = 0; p < NP; ++p)
        pv[p][u] = *(const float4*)(parts + ((int64_t)p * M + row) * N + 4 * lane + 256 * u);
      if (pbias) pb[u] = *(const half4_t*)(pbias + 4 * lane + 256 * u);
    }
  }
#pragma unroll
  for (int u = 0; u < NC; ++u) {
    wv[u] = *(const half4_t*)(w + 4 * lane + 256 * u);
    bv[u] = *(const half4_t*)(b + 4 * lane + 256 * u);
  }
  float v[NC][4];
  float s = 0.f;
#pragma unroll
  for (int u = 0; u < NC; ++u) {
    half4_t h = xv[u];
    if (NP > 0) {
      float a[4] = {pv[0][u].x, pv[0][u].y, pv[0][u].z, pv[0][u].w};
#pragma unroll
      for (int p = 1; p < NP; ++p) {
        a[0] += pv[p][u].x; a[1] += pv[p][u].y; a[2] += pv[p][u].z; a[3] += pv[p][u].w;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const half_t lin = pbias ? (half_t)(a[e] + (float)pb[u][e]) : (half_t)a[e];
        h[e] = (half_t)((float)h[e] + (float)lin);
      }
      *(half4_t*)(x_out + (int64_t)row * ldxo + 4 * lane + 256 * u) = h;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[u][e] = (float)h[e];
      s += v[u][e];
    }
  }
  const float mean = wave_sum(s) / (float)N;
  float q = 0.f;
#pragma unroll
  for (int u = 0; u < NC; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = v[u][e] - mean;
      q += d * d;
    }
  const float var = wave_sum(q) / (float)N;
  const float rstd = rsqrtf(var + eps);
#pragma unroll
  for (int u = 0; u < NC; ++u) {
    half4_t y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (half_t)((v[u][e] - mean) * rstd * (float)wv[u][e] + (float)bv[u][e]);
    *(half4_t*)(out + (int64_t)row * ldo + 4 * lane + 256 * u) = y;
  }
}

typedef void (*layernorm4_fn)(const half_t*, int, const half_t*, const half_t*, int, float,
                              half_t*, int, const float*, const half_t*, half_t*, int);
// The layernorm4_kernel instance for (N, nparts), or nullptr (the kernel above then).
static layernorm4_fn layernorm4_for(int N, int nparts) {
  if (N != 1280) return nullptr;
  switch (nparts) {
    case 0: return layernorm4_kernel<5, 0>;
    case 1: return layernorm4_kernel<5, 1>;
    case 2: return layernorm4_kernel<5, 2>;
    case 3: return layernorm4_kernel<5, 3>;
    case 4: return layernorm4_kernel<5, 4>;
  }
  return nullptr;
}

// LayerNorm of M rows of N (N % 8 == 0, N <= 2048); w, b fp16 [N]; out may alias x.
extern "C" int omni_layernorm(const void* x, int ldx, const void* weight, const void* bias, int M,
                              int N, float eps, void* out, int ldo, void* stream) {
  if (M < 0 || N <= 0) return OMNI_EINVAL;
  if (M == 0) return OMNI_OK;
  if ((N & 7) || N > 64 * 8 * LN_MAXCH) return OMNI_EUNSUPPORTED;
  if (!x || !weight || !bias || !out) return OMNI_EINVAL;
  if (ldx < N || ldo < N || (ldx & 7) || (ldo & 7)) return OMNI_EINVAL;
  if (layernorm4_fn kern = ((((uintptr_t)x | (uintptr_t)out | (uintptr_t)weight | (uintptr_t)bias) & 7) == 0 &&
                             (ldx & 3) == 0 && (ldo & 3) == 0) ? layernorm4_for(N, 0) : nullptr)
    hipLaunchKernelGGL(kern, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
                       (const half_t*)x, ldx, (const half_t*)weight, (const half_t*)bias, M, eps,
                       (half_t*)out, ldo, nullptr, nullptr, nullptr, 0);
  else
    hipLaunchKernelGGL(layernorm_kernel<false>, dim3((unsigned)((M + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, (const half_t*)x, ldx, (const half_t*)weight,
                       (const half_t*)bias, M, N, eps, (half_t*)out, ldo, nullptr, 0, nullptr,
                       nullptr, 0);
  OMNI_CHECK_LAUNCH();
  return OMNI_OK;
}

// The residual add of a split-K linear (fp32 slices [nparts][M][N], 1 <= nparts <= 16,
// optional fp16 bias [N]) followed by a LayerNorm: residual_out = fp16(residual +
// fp16(sum of the slices + bias)), as the linear's finish launch with the residual epilogue
// writes it, then out = LayerNorm(residual_out) as omni_layernorm (model/qwen2_vit.py:66-69:
// x = x + attn(...); norm2(x), and x = x + mlp(...) before the next block's norm1 or the
// merger's ln_q).  residual_out may alias residual.
extern "C" int omni_layernorm_partials(const float* partials, int nparts, const void* lin_bias,
                                       const void* residual, int ldr, void* residual_out, int ldro,
                                       const void* weight, const void* bias, int M, int N,
                                       float eps, void* out, int ldo, void* stream) {
  if (M < 0 || N <= 0 || nparts < 1 || nparts > 16) return OMNI_EINVAL;
  if (M == 0) return OMNI_OK;
  if ((N & 7) || N > 64 * 8 * LN_MAXCH) return OMNI_EUNSUPPORTED;
  if (!partials || !residual || !residual_out || !weight || !bias || !out) return OMNI_EINVAL;
  if (ldr < N || ldro < N || ldo < N || (ldr & 7) || (ldro & 7) || (ldo & 7)) return OMNI_EINVAL;
  if (((uintptr_t)partials & 15) || ((uintptr_t)residual & 15) || ((uintptr_t)residual_out & 15) ||
      ((uintptr_t)out & 15) || (lin_bias && ((uintptr_t)lin_bias & 15)))
    return OMNI_EINVAL;
  if (layernorm4_fn kern = (((uintptr_t)weight | (uintptr_t)bias) & 7) == 0 ? layernorm4_for(N, nparts) : nullptr)
    hipLaunchKernelGGL(kern, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
                       (const half_t*)residual, ldr, (const half_t*)weight, (const half_t*)bias, M,
                       eps, (half_t*)out, ldo, partials, (const half_t*)lin_bias,
                       (half_t*)residual_out, ldro);
  else
    hipLaunchKernelGGL(layernorm_kernel<true>, dim3((unsigned)((M + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, (const half_t*)residual, ldr, (const half_t*)weight,
                       (const half_t*)bias, M, N, eps, (half_t*)out, ldo, partials, nparts,
                       (const half_t*)lin_bias, (half_t*)residual_out, ldro);
  OMNI_CHECK_LAUNCH();
  return OMNI_OK;
}

// ---------------------------------------------------------------------------
// 2-D vision rotary, in place on the q and k heads of the qkv rows.
// For head_dim D (half R = D / 2, quarter R / 2): pair (d, d + R), d < R, is rotated by
//   angle_d = pos_h * inv_freq[d]        (d < R/2)
//           = pos_w * inv_freq[d - R/2]  (R/2 <= d < R)
// (model/qwen2_vit.py:96-116: freqs[pos_ids].flatten(1), emb = cat(rpe, rpe)), in fp32:
//   y[d] = x[d] cos - x[d+R] sin,  y[d+R] = x[d+R] cos + x[d] sin
// (kernels/vision_rope.py:19-24), rounded to fp16.  One thread per 8 consecutive d of one
// (token, q|k, head).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void vision_rope_kernel(half_t* __restrict__ qkv, int ld, int S,
                                                          int nh, int hd,
                                                          const int* __restrict__ pos_hw,
                                                          const float* __restrict__ inv_freq) {
#pragma clang fp contract(off)
  const int R = hd >> 1, Q = hd >> 2;
  const int cpr = R >> 3;                                // chunks per rotated half
  const int64_t total = (int64_t)S * 2 * nh * cpr;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int c = (int)(i % cpr);
  const int64_t r = i / cpr;
  const int head = (int)(r % (2 * nh));                  // q heads, then k heads
  const int t = (int)(r / (2 * nh));
  half_t* p = qkv + (int64_t)t * ld + head * hd + c * 8;
  const half8_t x1 = *(const half8_t*)p;
  const half8_t x2 = *(const half8_t*)(p + R);
  const float ph = (float)pos_hw[2 * t], pw = (float)pos_hw[2 * t + 1];
  half8_t y1, y2;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int d = c * 8 + e;
    const float ang = d < Q ? ph * inv_freq[d] : pw * inv_freq[d - Q];
    const float cs = cosf(ang), sn = sinf(ang);
    const float a = (float)x1[e], b = (float)x2[e];
    y1[e] = (half_t)(a * cs - b * sn);
    y2[e] = (half_t)(b * cs + a * sn);
  }
  *(half8_t*)p = y1;
  *(half8_t*)(p + R) = y2;
}

// Rotate q (heads [0, nh)) and k (heads [nh, 2 nh)) of S rows of qkv (row stride ld, head
// dim hd, hd % 16 == 0) in place.  pos_hw int32 [S][2] = (h, w) patch position;
// inv_freq fp32 [hd / 4].
extern "C" int omni_vision_rope(void* qkv, int ld, int S, int n_heads, int head_dim,
                                const int* pos_hw, const float* inv_freq, void* stream) {
  if (S < 0 || n_heads <= 0 || head_dim <= 0) return OMNI_EINVAL;
  if (S == 0) return OMNI_OK;
  if (head_dim & 15) return OMNI_EUNSUPPORTED;
  if (!qkv || !pos_hw || !inv_freq) return OMNI_EINVAL;
  if (ld < 2 * n_heads * head_dim || (ld & 7)) return OMNI_EINVAL;
  const int64_t total = (int64_t)S * 2 * n_heads * (head_dim / 16);
  const int64_t grid = (total + 255) / 256;
  if (grid > 0x7fffffff) return OMNI_EUNSUPPORTED;
  hipLaunchKernelGGL(vision_rope_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                     (half_t*)qkv, ld, S, n_heads, head_dim, pos_hw, inv_freq);
  OMNI_CHECK_LAUNCH();
  return OMNI_OK;
}

// ---------------------------------------------------------------------------
// Segmented non-causal attention, head_dim 80 (model/qwen2_vit.py:48-64): for every head
// and every query t of segment [cu[s], cu[s+1]), out[t] = softmax(q_t K^T * scale) V over
// the keys of the same segment.
//
// The 32-row tiles of attn_rows.h at 80 dims: 5 steps of 16 dims for the scores (nothing
// padded) and three 32-dim output blocks, the third's upper 16 rows computed from whatever
// follows a V row in LDS and never stored.  A workgroup owns 32 R consecutive queries of one
// segment and one head, its key tiles dealt to S groups of R waves whose states merge in LDS.
// K and V rows stay 160 bytes apart: the score operand's 16 rows x 16 bytes then repeat their
// banks every 8 rows, which a chunk swizzle by (row / 8) % 2 undoes, and the transposed V
// reads share banks in one row pair of four.
// The workgroups of one head are contiguous in the XCD-aware order, so that a head's K
// and V are read into one XCD's L2.
// MI355X, us per launch of 16 heads, 64 rows in 4 key groups / 128 rows in 2, then 16-row
// tiles: 1024 patches 14.2 / 17.5, 21.1; 600 10.0 / 12.7, 14.0; 500 + 260 + 700 19.2 / 14.7,
// 27.5; 2048 44.4 / 33.5, 71.4; 2852 + 1020 95.4 / 80.9 (580 TFLOP/s), 161.4.  128 rows read
// each staged tile twice as often and halve its traffic, but make half the workgroups: 64 rows
// while those fit one round of the CUs.  (One key group of 128 rows is 3-7 % faster on the
// large images and its error against 64 bits 1.6 % larger than the 16-row tiles': not used.)
// ---------------------------------------------------------------------------
#define VA_HD 80
#define VA_CPR 10      // 16-byte chunks per 80-dim row
#define VA_ROWB 160    // bytes per LDS row

struct VitAttnArgs {
  const half_t* qkv;   // rows [S][ld]: q heads | k heads | v heads, head_dim 80
  int ld;
  const int* cu;       // [nseg + 1]
  const int* tiles;    // [ntiles][2] = (first query, segment)
  int ntiles, nh, S;
  half_t* out;         // [S][ldo], head h at column 80 h
  int ldo;
  float scale_log2;    // > 0
  int negate;          // the scale was negative: its sign goes to q
};

// ALIGNED: qkv and out on 16-byte boundaries, ldo a multiple of 8, ld within the 32-bit lane
// offsets (tiles straight to LDS, 16-byte stores); otherwise staged through registers and stored
// by element.
template <int R, int S, int KT, bool ALIGNED>
__global__ __launch_bounds__(64 * R * S, 2) void vit_attn_kernel(VitAttnArgs a) {
  constexpr int NB = KT / 32;
  constexpr int TB = KT * VA_ROWB;                   // bytes of a K (or V) tile
  constexpr int NI = 2 * KT * VA_CPR / 64;           // 1 KB pieces of a K + V tile
  constexpr int NW = (NI + R - 1) / R;               // pieces per wave
  constexpr int NBUF = 2;
  static_assert(2 * KT * VA_CPR % 64 == 0 && TB % 1024 == 0, "tiles are whole 1 KB pieces");
  constexpr int MB = R * S * 40 * 64 * 4;            // the merge's outputs
  constexpr int LB = S * NBUF * 2 * TB + 64;         // + what the last row's third block reads
  __shared__ __attribute__((aligned(16))) char smem[LB > MB ? LB : MB];
  __shared__ float ml_lds[S][R][2][32];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / R;                          // key group
  const int rt = wave - grp * R;                     // row tile
  const int l32 = lane & 31, hf = lane >> 5;
  const int L = xcd_logical_block(blockIdx.x, gridDim.x);
  const int h = L / a.ntiles, tile = L - h * a.ntiles;
  const int q0 = a.tiles[2 * tile], seg = a.tiles[2 * tile + 1];
  const int beg = max(a.cu[seg], 0), end = min(a.cu[seg + 1], a.S);
  if (q0 < beg || q0 >= end) return;                 // malformed table entry: nothing to do
  const int nrows = min(end - q0, 32 * R);
  const bool rows_here = 32 * rt < nrows;
  const int row = min(32 * rt + l32, nrows - 1);

  half8_t qf[5];
  {
    const half_t* qp = a.qkv + (int64_t)(q0 + row) * a.ld + h * VA_HD + 8 * hf;
#pragma unroll
    for (int ks = 0; ks < 5; ++ks) {
      qf[ks] = *(const half8_t*)(qp + 16 * ks);
      if (a.negate) qf[ks] = -qf[ks];
    }
  }

  const int ntile = (end - beg + KT - 1) / KT;
  const int steps = (ntile + S - 1) / S;
  const int tbeg = grp * steps;
  const int nt = min(steps, ntile - tbeg);           // may be <= 0

  // piece J of a tile (J < NI / 2: K, else V): chunk c = 64 (J mod NI / 2) + lane is key
  // c / 10, 16-byte chunk c % 10, the K chunks swizzled in the source address
  uint32_t psrc[NW];
  int prow[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int J = rt + R * i;
    const bool is_v = J >= NI / 2;
    const int c = 64 * (is_v ? J - NI / 2 : J) + lane;
    prow[i] = c / VA_CPR;
    const int ch = c - prow[i] * VA_CPR;
    psrc[i] = (is_v ? 2u : 1u) * a.nh * (VA_HD * 2) + 16 * (is_v ? ch : ch ^ ((prow[i] >> 3) & 1));
  }
  const half_t* hbase = a.qkv + h * VA_HD;
  auto stage = [&](int kb, char* dst) {
    const half_t* src = hbase + (int64_t)kb * a.ld;
    const int last = end - 1 - kb;                   // the last tile repeats the last key
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int J = rt + R * i;
      if (NI % R && J >= NI) continue;
      if constexpr (ALIGNED)
        dma16(src, (uint32_t)min(prow[i], last) * (uint32_t)a.ld * 2 + psrc[i],
              __builtin_amdgcn_readfirstlane(lds_offset(dst)) + 1024 * J);
      else
        *(half8_t*)(dst + 1024 * J + 16 * lane) =
            *(const half8_t*)((const char*)(src + (int64_t)min(prow[i], last) * a.ld) + psrc[i]);
    }
  };

  float m_run = -INFINITY, l_run = 0.f;
  f32x16 o[3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  const int koff = l32 * VA_ROWB + ((hf ^ ((l32 >> 3) & 1)) << 4);
  const int i16 = lane & 15;
  const int voff = (4 * hf + (i16 >> 2)) * VA_ROWB + ((lane >> 4) & 1) * 32 + (i16 & 3) * 8;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

  char* gbuf = smem + grp * NBUF * 2 * TB;
  if (nt > 0) stage(beg + tbeg * KT, gbuf);
  // Q has landed (the compiler would otherwise count its loads as outstanding in the loop)
  __builtin_amdgcn_s_waitcnt(0x0f70);
  for (int it = 0; it < steps; ++it) {
    const char* kt = gbuf + (it & 1) * 2 * TB;
    const char* vt = kt + TB;
    const int kb = beg + (tbeg + it) * KT;
    vm_wait();             // this wave's pieces of tile it have landed; so, past the barrier,
    lds_barrier();         // have the others', and tile it - 1's buffer is free
    if (it + 1 < nt) stage(kb + KT, gbuf + ((it + 1) & 1) * 2 * TB);
    if (it >= nt || !rows_here) continue;
    f32x16 s[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[b][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 5; ++ks)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        s[b] = mfma32x32x16(*(const half8_t*)(kt + 32 * VA_ROWB * b + koff + 32 * ks), qf[ks], s[b]);
    if (kb + KT > end) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (kb + 32 * b + 8 * (i >> 2) + 4 * hf + (i & 3) >= end) s[b][i] = -INFINITY;
    }
    half8_t p[2 * NB];
    softmax32<NB, 3>(s, a.scale_log2, m_run, l_run, o, p);
#pragma unroll
    for (int t = 0; t < 2 * NB; ++t)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const char* vp = vt + 16 * VA_ROWB * t + voff + 64 * d;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)vp);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vp + 8 * VA_ROWB));
        const half4_t a0 = __builtin_bit_cast(half4_t, lo), a1 = __builtin_bit_cast(half4_t, hi);
        o[d] = mfma32x32x16((half8_t){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]},
                            p[t], o[d]);
      }
  }

  // The 10 output quads (lane half hf: dims 8 quad + 4 hf .. + 3), merged over the groups;
  // group g finishes quad pairs g, g + S, ..
  {
    float x, y;
    half_pair(l_run, x, y);
    l_run = x + y;
  }
  float* om = (float*)smem;
  __syncthreads();
  if (rows_here) {
#pragma unroll
    for (int q = 0; q < 10; ++q)
      *(float4*)(om + (((grp * R + rt) * 10 + q) * 64 + lane) * 4) =
          make_float4(o[q >> 2][4 * (q & 3)], o[q >> 2][4 * (q & 3) + 1], o[q >> 2][4 * (q & 3) + 2],
                      o[q >> 2][4 * (q & 3) + 3]);
    if (hf == 0) {
      ml_lds[grp][rt][0][l32] = m_run;
      ml_lds[grp][rt][1][l32] = l_run;
    }
  }
  __syncthreads();
  if (!rows_here) return;
  float M = ml_lds[0][rt][0][l32];                   // the first group is never empty
#pragma unroll
  for (int s = 1; s < S; ++s) M = fmaxf(M, ml_lds[s][rt][0][l32]);
  float f[S], den = 0.f;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    f[s] = __builtin_amdgcn_exp2f(ml_lds[s][rt][0][l32] - M);
    den += ml_lds[s][rt][1][l32] * f[s];
  }
  const float inv = 1.0f / den;
  half_t* op = a.out + (int64_t)(q0 + row) * a.ldo + h * VA_HD;
  const bool mine = 32 * rt + l32 < nrows;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    if (k % S != grp) continue;
    unsigned w[2][2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int q = 2 * k + e;
      float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const float4 v = *(const float4*)(om + (((s * R + rt) * 10 + q) * 64 + lane) * 4);
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
    // exchanged between the lane halves: half 0 has all 8 dims of quad 2 k, half 1 of 2 k + 1
    const auto r0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
    const auto r1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
    const u32x4 st = {r0[0], r1[0], r0[1], r1[1]};
    if (mine) {
      half_t* dp = op + 8 * (2 * k + hf);
      if constexpr (ALIGNED) {
        *(u32x4*)dp = st;
      } else {
        const half8_t hv = __builtin_bit_cast(half8_t, st);
#pragma unroll
        for (int e = 0; e < 8; ++e) dp[e] = hv[e];
      }
    }
  }
}

// Non-causal attention within segments over the qkv rows (q | k | v heads, head_dim 80,
// row stride ld), already rotated.  cu int32 [nseg + 1] (cu[0] = 0, increasing, cu[nseg]
// = S); tiles int32 [ntiles][2] = (first query, segment) covering every segment in steps
// of `rows` = 64 or 128 queries; out fp16 [S][ldo] (head h at column 80 h).
extern "C" int omni_vit_attention_rows(const void* qkv, int ld, int S, int n_heads, int head_dim,
                                       const int* cu_seqlens, const int* tiles, int ntiles,
                                       void* out, int ldo, float scale, int rows, void* stream) {
  if (S < 0 || n_heads <= 0 || ntiles < 0) return OMNI_EINVAL;
  if (rows != 64 && rows != 128) return OMNI_EINVAL;
  if (head_dim != VA_HD) return OMNI_EUNSUPPORTED;
  if (S == 0 || ntiles == 0) return OMNI_OK;
  if (!qkv || !cu_seqlens || !tiles || !out) return OMNI_EINVAL;
  if (ld < 3 * n_heads * VA_HD || (ld & 7) || ldo < n_heads * VA_HD) return OMNI_EINVAL;
  const int64_t grid = (int64_t)ntiles * n_heads;
  if (grid > 0x7fffffff) return OMNI_EUNSUPPORTED;
  VitAttnArgs a;
  a.qkv = (const half_t*)qkv;
  a.ld = ld;
  a.cu = cu_seqlens;
  a.tiles = tiles;
  a.ntiles = ntiles;
  a.nh = n_heads;
  a.S = S;
  a.out = (half_t*)out;
  a.ldo = ldo;
  a.scale_log2 = fabsf(scale) * 1.4426950408889634f;
  // A masked score times 0 would be NaN.  2^-126 weighs the keys as 0 does: fp16 heads' scores
  // are below 2^40, so every exponent is under 2^-86 and every exp2 exactly 1.
  if (a.scale_log2 < 0x1p-126f) a.scale_log2 = 0x1p-126f;
  a.negate = scale < 0.f;
  // a staged tile spans 64 rows of 2 ld bytes: below 2^32 up to ld = 2^24
  const bool al = (((uintptr_t)qkv | (uintptr_t)out) & 15) == 0 && (ldo & 7) == 0 && ld <= 1 << 24;
  const dim3 gd((unsigned)grid);
  hipStream_t st = (hipStream_t)stream;
  const dim3 bd(512);
  if (rows == 128) {
    if (al) hipLaunchKernelGGL((vit_attn_kernel<4, 2, 64, true>), gd, bd, 0, st, a);
    else hipLaunchKernelGGL((vit_attn_kernel<4, 2, 64, false>), gd, bd, 0, st, a);
  } else {
    if (al) hipLaunchKernelGGL((vit_attn_kernel<2, 4, 32, true>), gd, bd, 0, st, a);
    else hipLaunchKernelGGL((vit_attn_kernel<2, 4, 32, false>), gd, bd, 0, st, a);
  }
  OMNI_CHECK_LAUNCH();
  return OMNI_OK;
}

// omni_vit_attention_rows with tiles of 64 queries.
extern "C" int omni_vit_attention(const void* qkv, int ld, int S, int n_heads, int head_dim,
                                  const int* cu_seqlens, const int* tiles, int ntiles, void* out,
                                  int ldo, float scale, void* stream) {
  return omni_vit_attention_rows(qkv, ld, S, n_heads, head_dim, cu_seqlens, tiles, ntiles, out,
                                 ldo, scale, 64, stream);
}
