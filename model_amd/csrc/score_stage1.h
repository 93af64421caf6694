// What the stage-1 kernels share (score_select.hip, score_sort.hip): their
// parameters and the queries' MFMA operand.
#pragma once

#include "common.h"
#include "layout.h"
#include "mfma.h"

namespace mpl {

constexpr int kQueriesPerWave = 32;

struct ScoreParams {
  const void* q_hat;    // [M, HC, half]: normalised in the scoring type (mode 0) or raw fp32
  const float* q_len;   // [M, HC] or null (mode 0 input)
  float* out_qlen;      // [M, HC] or null (mode 2 output)
  int query_mode;       // MPL_Q_NORMALIZED / MPL_Q_RAW / MPL_Q_RAW_SCALED
  const uint4* packed;  // packed keys
  const float* gumbel;  // [M, HC, n] or null
  const float* T;           // device scalar: the clamped temperature
  const float* noise_coef;  // device scalar routing_noise * noise_scale (read with noise only)
  int noise_vec;  // gumbel rows 16-byte aligned (base aligned, n % 4 == 0)
  int64_t M;
  int HC, n, half, k, nblk, splits, blk_per_split;
  int pass1_blocks;  // blocks of each split scanned by the bound pass
  float* out_sel;    // [splits, M, HC, k] (null without noise: equals clean)
  float* out_clean;  // [splits, M, HC, k]
  int* out_idx;      // [splits, M, HC, k]
};

// The wave's MFMA query operand: lane l holds query row my_q (= the wave's
// first query + l % 32), dims 16c + 8*(l/32) + [0,8) of chunk c (fp16; the
// fp32 tile's map for fp32), and ql, the row's length factor (1 without
// query_scale / q_len).  Rows out of range (!valid) are zeros.  With
// write_qlen, mode RAW_SCALED also stores ql to out_qlen.
template <typename T, int NCH>
__device__ __forceinline__ void query_operand(const ScoreParams& p, int hc, int64_t my_q, bool valid, int lane,
                                              bool write_qlen, typename Mfma<T>::Op (&qop)[NCH], float& ql) {
  const int par = lane >> 5;
  ql = 1.f;
  if (p.query_mode == MPL_Q_NORMALIZED) {
    const T* qrow = (const T*)p.q_hat + (valid ? (my_q * p.HC + hc) * (int64_t)p.half : 0);
#pragma unroll
    for (int c = 0; c < NCH; ++c) qop[c] = Mfma<T>::load_q(qrow, valid, p.half, c, lane);
    if (p.q_len != nullptr) ql = p.q_len[(valid ? my_q : 0) * p.HC + hc];
  } else {
    // Raw fp32 queries, normalised here (memory.py:30-31, 136-137): the
    // lane pair holds the row's 2*NCH*8 dims, so one half-swap completes
    // the sum of squares.
    const float* qrow = (const float*)p.q_hat + (valid ? (my_q * p.HC + hc) * (int64_t)p.half : 0);
    float x[NCH][Mfma<T>::kQElems];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) Mfma<T>::load_q_raw(qrow, valid, p.half, c, lane, x[c], ss);
    float a = ss, b = ss;
    half_swap(a, b);
    const float tot = ss + (par ? a : b) + 1e-6f;
    const float rn = 1.0f / sqrtf(tot);
#pragma unroll
    for (int c = 0; c < NCH; ++c) qop[c] = Mfma<T>::scale_q(x[c], rn);
    if (p.query_mode == MPL_Q_RAW_SCALED) {
      ql = sqrtf(tot) / sqrtf((float)p.half);
      if (p.out_qlen != nullptr && valid && write_qlen && par == 0) p.out_qlen[my_q * p.HC + hc] = ql;
    }
  }
}

// Stage 1 by sorting (score_sort.hip): k <= kmax (16 or 32), no noise.  Its
// workgroups are single waves of 32 queries, so the grid has
// cdiv(M, 32) * splits * HC of them.  MPL_EUNSUPPORTED for an unknown HP.
int launch_score_sort(const ScoreParams& sp, int score_dtype, int HP, int kmax, hipStream_t s);

}  // namespace mpl
