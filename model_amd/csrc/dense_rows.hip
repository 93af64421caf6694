// Dense layers of the backbone for many rows (a whole sequence batch), up to
// three of the same input in one launch, with what surrounds them in
// model.py:29-127 fused in:
//
//   a     = x [rows, K] fp32;  a = LayerNorm(a) if ln_scale;  a = a * x_mul
//   out_i = act_i(a . W_i + bias_i) (+ residual)
//
// W_i is [K, N_i] (a Dense kernel) or [N_i, K] (the embedding table).  A
// workgroup of 4 waves owns a 64 x 64 tile of one layer's output, each wave a
// 32 x 32 block on v_mfma_f32_32x32x2_f32.  K runs in chunks of 32 through
// LDS: the next chunk's 16-byte loads are in flight while this one's MFMAs
// run.  The contraction is permuted so that one 16-byte LDS read of a row
// feeds four MFMAs (lanes of half h take dims 4h .. 4h+3 of each 8), for x
// and for [N, K] weights; [K, N] weights are read as they lie, one dword a
// MFMA.  LayerNorm statistics (mean, then the centred variance) are wave sums
// over the tile's own rows before the first chunk.  One order of the sums for
// every tile, so results do not depend on which layers share a launch.
//
// Bound: the fp32 MFMAs (64 cycles each, 16 a wave and chunk) at two thirds of
// their rate; what it saves are the passes around a product.  Measured, 4,096
// rows, us (the library's product alone): K = 256, N = 768 with LayerNorm 31.1
// (23.5), N = 256 11.5 (9.6), K = 1,024, N = 256 31.0 (21.7); a separate
// LayerNorm takes 8, each elementwise pass 4 to 10, and the whole backbone
// over 16 x 256 tokens goes from 1,490 to 935 with causal_attn.hip.  Chunks of
// 64 columns, two register sets of chunks in flight, 16x16x4 MFMAs and two
// groups of waves splitting K measured no faster.
#include <math.h>

#include "common.h"
#include "topk.h"

namespace mpl {
namespace {

constexpr int kTM = 64, kTN = 64, kKC = 32;
constexpr int kPA = kKC + 4;  // LDS pitch of row-major operands (16-byte rows, no bank conflicts)
constexpr int kPW = kTN + 8;  // LDS pitch of a [K, N] weight chunk: the lane halves' rows, 4 apart, fall 32 banks apart
constexpr int kMaxLayers = 3;

struct DenseLayer {
  const float* w;
  const float* bias;
  float* out;
  int64_t pitch;
  int N, act, tile0;  // tile0: the layer's first column tile in the grid
};

struct DenseArgs {
  const float* x;
  const float* x_mul;
  const float* ln_scale;
  const float* ln_bias;
  const float* residual;  // one layer only, its output's shape
  int64_t rows;
  int K, count;
  float eps;
  DenseLayer layer[kMaxLayers];
};

__device__ __forceinline__ float activate(float v, int act) {
  if (act == MPL_ACT_GELU_TANH) {
    const float inner = 0.7978845608028654f * (v + 0.044715f * v * v * v);
    return 0.5f * v * (1.0f + tanhf(inner));
  }
  if (act == MPL_ACT_SILU) return v / (1.0f + expf(-v));
  return v;
}

// Sums of 16 values over the wave's 64 lanes, scattered: lane l ends with the
// sums of values i + 4 * ((l >> 4) & 1) + 8 * (l >> 5) in v[i], i < 4.  Two
// swapping steps halve the values a lane holds before the four 16-lane ones
// (40 instructions; summing all 16 in every lane took four times that and
// 4 us of a launch).
__device__ __forceinline__ void wave_sums16(float (&v)[16], int lane) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    half_swap(v[i], v[i + 8]);
    v[i] += v[i + 8];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 4]), false, false);
    v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#define MPL_STEP(S)                                     \
  _Pragma("unroll") for (int i = 0; i < 4; ++i) v[i] += \
      __uint_as_float(w64::xr<S>(__float_as_uint(v[i]), lane));
  MPL_STEP(1) MPL_STEP(2) MPL_STEP(4) MPL_STEP(8)
#undef MPL_STEP
}

// Zeroes a loaded vector where !ok, by bits: a select of a loaded value would
// become a branch around its load.
__device__ __forceinline__ float4 keep_if(float4 v, bool ok) {
  const uint32_t m = ok ? 0xFFFFFFFFu : 0u;
  return make_float4(__uint_as_float(__float_as_uint(v.x) & m), __uint_as_float(__float_as_uint(v.y) & m),
                     __uint_as_float(__float_as_uint(v.z) & m), __uint_as_float(__float_as_uint(v.w) & m));
}

template <int LAYOUT, bool LN, bool MUL>
__global__ __launch_bounds__(256) void dense_rows_kernel(DenseArgs p) {
  __shared__ float sa[kTM * kPA];
  __shared__ float sw[LAYOUT == MPL_W_IN_OUT ? kKC * kPW : kTN * kPA];
  __shared__ float smean[kTM], srstd[kTM];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t m0 = (int64_t)blockIdx.y * kTM;
  int li = 0;
  if (p.count > 1 && (int)blockIdx.x >= p.layer[1].tile0) li = 1;
  if (p.count > 2 && (int)blockIdx.x >= p.layer[2].tile0) li = 2;
  const DenseLayer L = p.layer[li];
  const int n0 = ((int)blockIdx.x - L.tile0) * kTN;
  const int K = p.K;

  // Thread's 16-byte pieces of a chunk: of x, rows tid/16 + 16 i, columns
  // 4 (tid % 16); of W the same places of a [64][64] block.  Rows and columns
  // past the ends are read clamped; what lies past K is zeroed in both.
  constexpr int CA = kKC / 4, RA = 256 / CA, NA = kTM / RA;  // row-major operands: columns, rows a pass, passes
  constexpr int NW = LAYOUT == MPL_W_IN_OUT ? kKC / 16 : NA;
  const int pr = tid / CA, pc = 4 * (tid % CA);
  const int wr = LAYOUT == MPL_W_IN_OUT ? tid >> 4 : pr, wc = LAYOUT == MPL_W_IN_OUT ? 4 * (tid & 15) : pc;
  float4 ra[NA], rw[NW], rm[MUL ? NA : 1];
  auto fetch = [&](int k0) __attribute__((always_inline)) {
    const int kc = min(k0 + pc, K - 4);
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int64_t row = min(m0 + pr + RA * i, p.rows - 1);
      ra[i] = *(const float4*)(p.x + row * K + kc);
      if (MUL) rm[MUL ? i : 0] = *(const float4*)(p.x_mul + row * K + kc);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if (LAYOUT == MPL_W_IN_OUT)
        rw[i] = *(const float4*)(L.w + (int64_t)min(k0 + wr + 16 * i, K - 1) * L.N + min(n0 + wc, L.N - 4));
      else
        rw[i] = *(const float4*)(L.w + (int64_t)min(n0 + wr + RA * i, L.N - 1) * K + kc);
    }
  };
  fetch(0);

  if (LN) {
    // 16 rows a wave, all requested at once: one memory round trip for up to
    // 256 columns, which then stay in registers for the second pass
    const float inv = 1.f / (float)K;
    const float* src[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) src[i] = p.x + min(m0 + 16 * wave + i, p.rows - 1) * K;
    float4 t[16];
    float s[16], v[16];
    auto rows16 = [&](int c0) __attribute__((always_inline)) {
      const int c = c0 + 4 * lane;
#pragma unroll
      for (int i = 0; i < 16; ++i) t[i] = *(const float4*)(src[i] + min(c, K - 4));
    };
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = v[i] = 0.f;
    for (int c0 = 0; c0 < K; c0 += 4 * kWave) {
      rows16(c0);
      const bool ok = c0 + 4 * lane < K;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float4 u = keep_if(t[i], ok);
        s[i] += (u.x + u.y) + (u.z + u.w);
      }
    }
    wave_sums16(s, lane);
    const int row0 = 16 * wave + 4 * ((lane >> 4) & 1) + 8 * (lane >> 5);  // the lane's four rows
    if ((lane & 15) == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) smean[row0 + i] = s[i] * inv;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = smean[16 * wave + i];
    for (int c0 = 0; c0 < K; c0 += 4 * kWave) {
      if (K > 4 * kWave) rows16(c0);  // wave-uniform
      const bool ok = c0 + 4 * lane < K;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float4 u = keep_if(make_float4(t[i].x - s[i], t[i].y - s[i], t[i].z - s[i], t[i].w - s[i]), ok);
        v[i] += (u.x * u.x + u.y * u.y) + (u.z * u.z + u.w * u.w);
      }
    }
    wave_sums16(v, lane);
    if ((lane & 15) == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) srstd[row0 + i] = rsqrtf(v[i] * inv + p.eps);
    }
    __syncthreads();
  }

  auto stage = [&](int k0) __attribute__((always_inline)) {
    const bool kok = k0 + pc < K;
    const int kc = min(k0 + pc, K - 4);
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f), be = g;
    if (LN) {
      g = *(const float4*)(p.ln_scale + kc);
      be = *(const float4*)(p.ln_bias + kc);
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      float4 a = ra[i];
      if (LN) {
        const float mu = smean[pr + RA * i], rs = srstd[pr + RA * i];
        a = make_float4((a.x - mu) * rs * g.x + be.x, (a.y - mu) * rs * g.y + be.y, (a.z - mu) * rs * g.z + be.z,
                        (a.w - mu) * rs * g.w + be.w);
      }
      if (MUL) {
        const float4 q = rm[MUL ? i : 0];
        a = make_float4(a.x * q.x, a.y * q.y, a.z * q.z, a.w * q.w);
      }
      *(float4*)(sa + (pr + RA * i) * kPA + pc) = keep_if(a, kok);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if (LAYOUT == MPL_W_IN_OUT)
        *(float4*)(sw + (wr + 16 * i) * kPW + wc) = keep_if(rw[i], k0 + wr + 16 * i < K);
      else
        *(float4*)(sw + (wr + RA * i) * kPA + wc) = keep_if(rw[i], kok);
    }
  };

  const int col = lane & 31, h = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  const float* pa = sa + (32 * wm + col) * kPA + 4 * h;
  const float* pw = LAYOUT == MPL_W_IN_OUT ? sw + 4 * h * kPW + 32 * wn + col : sw + (32 * wn + col) * kPA + 4 * h;
  f32x16 acc = f32x16{};
  for (int k0 = 0; k0 < K; k0 += kKC) {
    if (k0 > 0) __syncthreads();  // every wave has read the chunk before
    stage(k0);
    __syncthreads();
    if (k0 + kKC < K) fetch(k0 + kKC);
    float4 a[kKC / 8], b[kKC / 8];  // the chunk's operands, requested before the first MFMA
#pragma unroll
    for (int g = 0; g < kKC / 8; ++g) {
      a[g] = *(const float4*)(pa + 8 * g);
      if (LAYOUT == MPL_W_IN_OUT)
        b[g] = make_float4(pw[(8 * g + 0) * kPW], pw[(8 * g + 1) * kPW], pw[(8 * g + 2) * kPW], pw[(8 * g + 3) * kPW]);
      else
        b[g] = *(const float4*)(pw + 8 * g);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < kKC / 8; ++g) {
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].x, b[g].x, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].y, b[g].y, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].z, b[g].z, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].w, b[g].w, acc, 0, 0, 0);
    }
  }

  const int n = n0 + 32 * wn + col;
  if (n >= L.N) return;
  const float bias = L.bias != nullptr ? L.bias[n] : 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t row = m0 + 32 * wm + 8 * (r >> 2) + 4 * h + (r & 3);
    if (row < p.rows) {
      float v = activate(acc[r] + bias, L.act);
      if (p.residual != nullptr) v += p.residual[row * L.N + n];
      L.out[row * L.pitch + n] = v;
    }
  }
}

template <int LAYOUT>
void launch_dense(const DenseArgs& a, dim3 grid, hipStream_t s) {
  const bool ln = a.ln_scale != nullptr, mul = a.x_mul != nullptr;
  if (ln && mul) dense_rows_kernel<LAYOUT, true, true><<<grid, 256, 0, s>>>(a);
  else if (ln) dense_rows_kernel<LAYOUT, true, false><<<grid, 256, 0, s>>>(a);
  else if (mul) dense_rows_kernel<LAYOUT, false, true><<<grid, 256, 0, s>>>(a);
  else dense_rows_kernel<LAYOUT, false, false><<<grid, 256, 0, s>>>(a);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace
}  // namespace mpl

using namespace mpl;

extern "C" int mpl_dense_layers(const float* x, const float* x_mul, const float* ln_scale, const float* ln_bias,
                                float ln_eps, int count, const void* weights, int weight_layout, const void* biases,
                                const void* widths, const void* activations, const float* residual, const void* outs,
                                const void* out_pitches, int64_t rows, int K, void* stream) {
  clear_error();
  MPL_REQUIRE(rows >= 0 && K >= 4 && K % 4 == 0 && count >= 1 && count <= kMaxLayers, MPL_EINVAL,
              "mpl_dense_layers: rows=%lld K=%d count=%d (K a positive multiple of 4, 1 to %d layers)", (long long)rows,
              K, count, kMaxLayers);
  MPL_REQUIRE(weight_layout == MPL_W_IN_OUT || weight_layout == MPL_W_OUT_IN, MPL_EINVAL,
              "mpl_dense_layers: bad weight_layout %d", weight_layout);
  MPL_REQUIRE((ln_scale == nullptr) == (ln_bias == nullptr), MPL_EINVAL,
              "mpl_dense_layers: ln_scale and ln_bias go together");
  MPL_REQUIRE(weights && biases && widths && activations && outs && out_pitches, MPL_EINVAL,
              "mpl_dense_layers: null table");
  MPL_REQUIRE(rows <= (int64_t)65535 * kTM, MPL_EINVAL, "mpl_dense_layers: rows=%lld above %d", (long long)rows,
              65535 * kTM);
  if (rows == 0) return MPL_OK;
  MPL_REQUIRE(x != nullptr, MPL_EINVAL, "mpl_dense_layers: null x");
  MPL_REQUIRE(aligned16(x) && aligned16(x_mul) && aligned16(ln_scale) && aligned16(ln_bias), MPL_EINVAL,
              "mpl_dense_layers: x, x_mul, ln_scale and ln_bias must be 16-byte aligned");
  MPL_REQUIRE(residual == nullptr || count == 1, MPL_EINVAL, "mpl_dense_layers: a residual goes with one layer");
  DenseArgs a{x, x_mul, ln_scale, ln_bias, residual, rows, K, count, ln_eps, {}};
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) {
    DenseLayer& L = a.layer[i];
    L.w = ((const float* const*)weights)[i];
    L.bias = ((const float* const*)biases)[i];
    L.out = ((float* const*)outs)[i];
    L.pitch = ((const int64_t*)out_pitches)[i];
    L.N = ((const int*)widths)[i];
    L.act = ((const int*)activations)[i];
    MPL_REQUIRE(L.N >= 4 && L.N % 4 == 0 && L.pitch >= L.N, MPL_EINVAL,
                "mpl_dense_layers: layer %d has width %d, pitch %lld (widths are positive multiples of 4)", i, L.N,
                (long long)L.pitch);
    MPL_REQUIRE(L.act == MPL_ACT_NONE || L.act == MPL_ACT_GELU_TANH || L.act == MPL_ACT_SILU, MPL_EINVAL,
                "mpl_dense_layers: bad activation %d", L.act);
    MPL_REQUIRE(L.w && L.out && aligned16(L.w), MPL_EINVAL, "mpl_dense_layers: layer %d: null or unaligned buffer", i);
    MPL_REQUIRE(L.out != x && L.out != x_mul, MPL_EINVAL, "mpl_dense_layers: out may alias residual only");
    L.tile0 = (int)tiles;
    tiles += cdiv(L.N, kTN);
  }
  MPL_REQUIRE(tiles < ((int64_t)1 << 31), MPL_EUNSUPPORTED, "mpl_dense_layers: too many columns");
  const dim3 grid((unsigned)tiles, (unsigned)cdiv(rows, kTM));
  if (weight_layout == MPL_W_OUT_IN) launch_dense<MPL_W_OUT_IN>(a, grid, (hipStream_t)stream);
  else launch_dense<MPL_W_IN_OUT>(a, grid, (hipStream_t)stream);
  return check_launch("mpl_dense_layers");
}
