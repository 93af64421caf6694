// Causal self-attention of whole sequences (model.py:88-95 outside decode
// mode: Flax MultiHeadDotProductAttention under a causal mask), forward only:
//
//   out[b, t, h, :] = softmax_{s <= t}((scale * q_t) . k_s) v_s
//
// from the fused projection qkv [batch, T, 3, heads, hd] fp32 (biases added).
// A workgroup of 4 waves owns 32 queries of one (sequence, head); wave w takes
// key blocks w, w + 4, ... of 32 keys up to the diagonal, with an online
// softmax, and the four partial results meet in LDS.  The scores are the
// transposed tile K . Q^T on v_mfma_f32_32x32x2_f32: lanes l and l + 32 hold
// 16 keys each of query l % 32, so maxima and sums are lane-local but for one
// half-swap, and each score register is directly the K = 2 operand of the
// product with V (the two halves' keys are 4 apart), as in the balance
// kernels.  Keys and values go from L2 straight to the operands: no score
// matrix, mask, transposed copy or softmax pass over memory.
//
// Bound: the MFMAs, hd a key block and wave (64 cycles each); the split over
// key blocks keeps the longest wave at a quarter of the last query tile's.
// 16 sequences of 256 tokens, 4 heads of 64: 20.9 us a layer, against about
// 110 for two batched products, scale, mask, softmax and transposed copies.
#include <math.h>

#include "common.h"

namespace mpl {
namespace {

constexpr int kAW = 4;  // waves per workgroup

template <int HD>
__global__ __launch_bounds__(kAW * kWave) void causal_attention_kernel(const float* __restrict__ qkv, int T, int H,
                                                                      float scale, float* __restrict__ out) {
  constexpr int DT = HD / 32;  // 32-dim tiles of the output
  constexpr int PO = HD + 4;
  __shared__ float so[kAW][32][PO];
  __shared__ float sm[kAW][32], sl[kAW][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int q0 = blockIdx.x * 32;
  const int64_t b = blockIdx.y / H;
  const int h = blockIdx.y % H;
  const int64_t tok = 3 * (int64_t)H * HD;  // floats per token
  const float* base = qkv + b * T * tok + (int64_t)h * HD;
  const float* kb = base + (int64_t)H * HD;
  const float* vb = base + 2 * (int64_t)H * HD;
  const int qi = q0 + col;

  float4 q[HD / 8];
#pragma unroll
  for (int g = 0; g < HD / 8; ++g) {
    float4 t = *(const float4*)(base + (int64_t)min(qi, T - 1) * tok + 8 * g + 4 * half);
    q[g] = make_float4(t.x * scale, t.y * scale, t.z * scale, t.w * scale);
  }
  float m = -INFINITY, l = 0.f;
  f32x16 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = f32x16{};

  const int last = min(q0 + 31, T - 1) / 32;
  for (int j = wave; j <= last; j += kAW) {
    const int k0 = 32 * j;
    const float* krow = kb + (int64_t)min(k0 + col, T - 1) * tok + 4 * half;
    float4 kv[HD / 8];
#pragma unroll
    for (int g = 0; g < HD / 8; ++g) kv[g] = *(const float4*)(krow + 8 * g);
    float v[16][DT];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float* vrow = vb + (int64_t)min(k0 + 8 * (r >> 2) + 4 * half + (r & 3), T - 1) * tok + col;
#pragma unroll
      for (int d = 0; d < DT; ++d) v[r][d] = vrow[32 * d];
    }
    f32x16 s = f32x16{};
#pragma unroll
    for (int g = 0; g < HD / 8; ++g) {
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[g].x, q[g].x, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[g].y, q[g].y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[g].z, q[g].z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[g].w, q[g].w, s, 0, 0, 0);
    }
    if (j == last) {  // wave-uniform: the diagonal block (keys past T - 1 lie past every query too)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (k0 + 8 * (r >> 2) + 4 * half + (r & 3) > qi) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    float a0 = mx, a1 = mx;
    half_swap(a0, a1);
    mx = fmaxf(m, fmaxf(a0, a1));
    // a query's key k0 is never masked (k0 <= q0), so mx > -inf unless scores are -inf themselves
    const float ref = mx == -INFINITY ? 0.f : mx;
    const float alpha = expf(m - ref);
    m = mx;
    float sum = 0.f, pr[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      pr[r] = expf(s[r] - ref);
      sum += pr[r];
    }
    l = l * alpha + sum;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[d][r] *= alpha;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[r][d], pr[r], acc[d], 0, 0, 0);
    }
  }

  float l0 = l, l1 = l;
  half_swap(l0, l1);
  if (half == 0) {
    sm[wave][col] = m;
    sl[wave][col] = l0 + l1;
  }
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *(float4*)&so[wave][col][32 * d + 8 * (r >> 2) + 4 * half] =
          make_float4(acc[d][r], acc[d][r + 1], acc[d][r + 2], acc[d][r + 3]);
  __syncthreads();
  for (int i = tid; i < 32 * HD; i += kAW * kWave) {
    const int t = i / HD, d = i % HD;
    float mm = sm[0][t];
#pragma unroll
    for (int w = 1; w < kAW; ++w) mm = fmaxf(mm, sm[w][t]);
    const float ref = mm == -INFINITY ? 0.f : mm;
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < kAW; ++w) {
      const float f = expf(sm[w][t] - ref);  // 0 for a wave that had no block
      num += f * so[w][t][d];
      den += f * sl[w][t];
    }
    if (q0 + t < T) out[((b * T + q0 + t) * H + h) * (int64_t)HD + d] = num / den;
  }
}

}  // namespace
}  // namespace mpl

using namespace mpl;

extern "C" int mpl_causal_attention(const float* qkv, int64_t batch, int T, int heads, int head_dim, float scale,
                                    float* out, void* stream) {
  clear_error();
  MPL_REQUIRE(batch >= 0 && T >= 0 && heads > 0, MPL_EINVAL, "mpl_causal_attention: bad sizes batch=%lld T=%d heads=%d",
              (long long)batch, T, heads);
  MPL_REQUIRE(head_dim == 32 || head_dim == 64 || head_dim == 128, MPL_EUNSUPPORTED,
              "mpl_causal_attention: head_dim %d (32, 64 or 128)", head_dim);
  MPL_REQUIRE(batch * heads <= 65535, MPL_EUNSUPPORTED, "mpl_causal_attention: batch * heads = %lld above 65535",
              (long long)(batch * heads));
  if (batch == 0 || T == 0) return MPL_OK;
  MPL_REQUIRE(qkv && out, MPL_EINVAL, "mpl_causal_attention: null buffer");
  MPL_REQUIRE(((uintptr_t)qkv & 15) == 0, MPL_EINVAL, "mpl_causal_attention: qkv must be 16-byte aligned");
  MPL_REQUIRE(out != qkv, MPL_EINVAL, "mpl_causal_attention: out may not alias qkv");
  const dim3 grid((unsigned)cdiv(T, 32), (unsigned)(batch * heads));
  hipStream_t s = (hipStream_t)stream;
  if (head_dim == 32) causal_attention_kernel<32><<<grid, kAW * kWave, 0, s>>>(qkv, T, heads, scale, out);
  else if (head_dim == 64) causal_attention_kernel<64><<<grid, kAW * kWave, 0, s>>>(qkv, T, heads, scale, out);
  else causal_attention_kernel<128><<<grid, kAW * kWave, 0, s>>>(qkv, T, heads, scale, out);
  return check_launch("mpl_causal_attention");
}
