// Attention on 32-row tiles: what the decoder's prefill (attn_rows.hip) and the vision
// tower's attention (vit.hip) share.
#pragma once

#include "common.h"

// ---------------------------------------------------------------------------
// One wave owns 32 query rows and walks key tiles with 32 x 32 x 16 MFMAs:
//   S^T [32 keys x 32 rows] = K . Q^T      (A = K rows from LDS, B = Q in registers)
//   O^T [32 dims x 32 rows] += V^T . P^T   (A = V read back transposed, B = P)
// In both products a lane's column is one query row (lane % 32), so the running maximum,
// the sum and the rescaling factor are per-lane scalars, and the scores' register layout
// is the B operand of the second product once the keys of a 16-key step are taken in the
// order the scores come in: register i of lane half h is key (i % 4) + 8 (i / 4) + 4 h.
//
// What bounds it is the vector unit beside the matrix cores: 64 keys x 32 rows are 32
// MFMAs of 32 cycles and, per lane, 32 scores through max, fma, exp2, add and the fp16
// conversion.  So per score there is nothing else: the scale rides in the fma, exp2 is the
// bare instruction (a result below 2^-126 reads 0, far under what fp16 P holds), keys are
// only masked in the tiles that cross a row's limit, and a tile that raises no row's maximum
// skips the 64 multiplies of the output.  (Skipping until a maximum has grown by 2^8 gained
// 2 % and cost accuracy: a row's largest P is then not exactly 1.)
// ---------------------------------------------------------------------------
__device__ __forceinline__ f32x16 mfma32x32x16(half8_t a, half8_t b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Lanes l and l + 32 exchanged: a = the lower half's value, b = the upper half's, in both
// halves.  In asm, with the wait states a swap needs after its operands are written: through
// the builtin the compiler takes the two results of equal operands for one value.
__device__ __forceinline__ void half_pair(float v, float& a, float& b) {
  a = v;
  b = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}

// One key tile's scores s (NB blocks of 32 keys) to probabilities p (the B operands of
// 2 NB 16-key steps), with the row state m_run (log2 units) and l_run (this lane half's part
// of the sum) updated and the NO output blocks rescaled where a maximum has moved.
template <int NB, int NO>
__device__ __forceinline__ void softmax32(const f32x16 (&s)[NB], float scale_log2, float& m_run,
                                          float& l_run, f32x16 (&o)[NO], half8_t (&p)[2 * NB]) {
  float mx = s[0][0];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[b][i]);
  float ma, mb;
  half_pair(mx, ma, mb);
  const float mt = fmaxf(ma, mb) * scale_log2;            // scale > 0: the scaled maximum
  if (__any(mt > m_run)) {
    const float m_new = fmaxf(m_run, mt);
    // -inf: a row none of whose keys has been seen (a key group that starts past its limit)
    const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int d = 0; d < NO; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
  }
  const float m_ref = m_run == -INFINITY ? 0.f : m_run;
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float e = __builtin_amdgcn_exp2f(fmaf(s[b][i], scale_log2, -m_ref));
      sum[i & 3] += e;
      p[2 * b + (i >> 3)][i & 7] = (half_t)e;
    }
  l_run += (sum[0] + sum[1]) + (sum[2] + sum[3]);
}

// 64 x 16 bytes global -> LDS: lane l's bytes at sbase + voff to LDS offset lds + 16 l.  In asm,
// with no register result: the compiler then counts nothing outstanding and does not make every
// LDS read that follows wait for the transfer; the reader waits itself (vm_wait + a barrier).
__device__ __forceinline__ void dma16(const void* sbase, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(sbase), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void vm_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}
