// Dense layers of the backbone for many rows (a whole sequence batch), up to
// three of the same input in one launch, with what surrounds them in
// model.py:29-127 fused in:
//
//   a     = x [rows, K] fp32;  a = LayerNorm(a) if ln_scale;  a = a * x_mul
//   out_i = act_i(a . W_i + bias_i) (+ residual)
//
// W_i is [K, N_i] (a Dense kernel) or [N_i, K] (the embedding table).  A
// workgroup of 4 waves owns a 64 x 64 tile of one layer's output, each wave a
// 32 x 32 block on v_mfma_f32_32x32x2_f32.  K runs in chunks of 32 through two
// LDS buffers: while a chunk's MFMAs run, the next one goes into the other
// buffer and the 16-byte loads of the one three later are sent (two register
// sets in flight), and the last four MFMAs cover the next chunk's LDS reads;
// one barrier a chunk.  The contraction is permuted so that one 16-byte LDS
// read of a row feeds four MFMAs (lanes of half h take dims 4h .. 4h+3 of each
// 8), for x and for [N, K] weights; [K, N] weights are read as they lie, one
// dword a MFMA.  LayerNorm statistics (mean, then the centred variance) are
// wave sums over the tile's own rows before the first chunk.  One order of the
// sums for every tile, so results do not depend on which layers share a launch.
//
// Bound: the fp32 MFMAs (64 cycles each, 16 a wave and chunk: 0.43 us), with
// 6 us of launch, first loads and epilogue around them and 5 us for LayerNorm.
// A chunk takes 0.56 us at one wave a SIMD; 0.47 without the staging between
// the MFMAs.  Measured, 4,096 rows, us, with one LDS buffer and one register
// set -> now: K = 256, N = 768 with LayerNorm 30.5 -> 27.1, N = 1,024 with
// LayerNorm and GELU 41.7 -> 37.6, N = 256 13.2 -> 11.5, K = 1,024, N = 256
// 34.2 -> 26.0.  Chunks of 64 columns, 16x16x4 MFMAs and two groups of waves
// splitting K measured no faster.
#include <math.h>

#include <type_traits>

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
  uint32_t tiles;  // column tiles of all the layers
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
__global__ __launch_bounds__(256, MUL ? 3 : 4) void dense_rows_kernel(DenseArgs p) {
  constexpr int SA = kTM * kPA, SW = LAYOUT == MPL_W_IN_OUT ? kKC * kPW : kTN * kPA;
  __shared__ float sa[2 * SA];
  __shared__ float sw[2 * SW];
  __shared__ float smean[kTM], srstd[kTM];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Workgroups go to the 8 XCDs in turn; each XCD takes a run of neighbouring
  // row tiles with all their column tiles, so its L2 holds an eighth of x.
  const uint32_t id = blockIdx.x, full = gridDim.x / 8 * 8;
  const uint32_t at = id < full ? (id & 7) * (full / 8) + (id >> 3) : id;
  const int64_t m0 = (int64_t)(at / p.tiles) * kTM;
  const int tile = (int)(at % p.tiles);
  int li = 0;
  if (p.count > 1 && tile >= p.layer[1].tile0) li = 1;
  if (p.count > 2 && tile >= p.layer[2].tile0) li = 2;
  const DenseLayer L = p.layer[li];
  const int n0 = (tile - L.tile0) * kTN;
  const int K = p.K;

  // Thread's 16-byte pieces of a chunk of 32 columns of K: of x, rows tid / 8 +
  // 32 i, columns 4 (tid % 8); of an [N, K] W the same places of a [64][32]
  // block, of a [K, N] W rows tid / 16 + 16 i, columns 4 (tid % 16) of a
  // [32][64] block.  Rows and columns past the ends are read clamped; what lies
  // past K is zeroed in both.
  constexpr int CA = kKC / 4, RA = 256 / CA, NA = kTM / RA;  // row-major operands: columns, rows a pass, passes
  constexpr int NW = LAYOUT == MPL_W_IN_OUT ? kKC / 16 : NA;
  const int pr = tid / CA, pc = 4 * (tid % CA);
  const int wr = LAYOUT == MPL_W_IN_OUT ? tid >> 4 : pr, wc = LAYOUT == MPL_W_IN_OUT ? 4 * (tid & 15) : pc;
  // These point at the thread's pieces of chunk `at_k` (which the main loop
  // advances); a chunk that may reach past K is read clamped.
  const float *xp[NA], *mp[MUL ? NA : 1], *wp[NW];
  int at_k = 0;
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int64_t row = min(m0 + pr + RA * i, p.rows - 1) * K;
    xp[i] = p.x + row + pc;
    if (MUL) mp[MUL ? i : 0] = p.x_mul + row + pc;
  }
#pragma unroll
  for (int i = 0; i < NW; ++i)
    wp[i] = LAYOUT == MPL_W_IN_OUT ? L.w + min(n0 + wc, L.N - 4) + (int64_t)(wr + 16 * i) * L.N
                                   : L.w + (int64_t)min(n0 + wr + RA * i, L.N - 1) * K + pc;
  // Whole: the main loop's addresses step along and nothing is masked (10 %
  // of a K = 1,024 layer).  Not with LayerNorm, whose registers would spill
  // (29.4 us against 27.5 at N = 768).
  using Yes = std::true_type;
  using No = std::false_type;
  using Whole = std::integral_constant<bool, !LN>;
  struct Pieces {
    float4 a[NA], w[NW], m[MUL ? NA : 1];
  };
  Pieces set0, set1;  // of two chunks, in flight
  float4 rg, rb;
  auto fetch = [&](Pieces& r, int k0, auto WHOLE) __attribute__((always_inline)) {
    const int kd = k0 - at_k;
    const int kc = WHOLE ? kd : min(k0 + pc, K - 4) - pc - at_k;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      r.a[i] = *(const float4*)(xp[i] + kc);
      if (MUL) r.m[MUL ? i : 0] = *(const float4*)(mp[MUL ? i : 0] + kc);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if (LAYOUT == MPL_W_IN_OUT)
        r.w[i] = *(const float4*)(wp[i] + (int64_t)((WHOLE ? k0 : min(k0, K - 1 - wr - 16 * i)) - at_k) * L.N);
      else
        r.w[i] = *(const float4*)(wp[i] + kc);
    }
  };
  auto fetch_ln = [&](int k0) __attribute__((always_inline)) {
    const int kc = min(k0 + pc, K - 4);
    rg = *(const float4*)(p.ln_scale + kc);
    rb = *(const float4*)(p.ln_bias + kc);
  };
  if (!LN) fetch(set0, 0, No{});

  if (LN) {
    // 16 rows a wave, all requested at once: one memory round trip for up to
    // 256 columns, which then stay in registers for the second pass
    const float inv = 1.f / (float)K;
    const float* src[16];
    const int w0 = 16 * __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
    for (int i = 0; i < 16; ++i) src[i] = p.x + min(m0 + w0 + i, p.rows - 1) * K;
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

  if (LN) {  // the statistics take the registers until here
    fetch(set0, 0, No{});
    fetch_ln(0);
  }
  fetch(set1, kKC, No{});  // past K: clamped, and not used
  float mu[NA], rs[NA];
#pragma unroll
  for (int i = 0; LN && i < NA; ++i) {
    mu[i] = smean[pr + RA * i];
    rs[i] = srstd[pr + RA * i];
  }
  auto stage = [&](const Pieces& r, int k0, int buf, auto WHOLE) __attribute__((always_inline)) {
    const bool kok = k0 + pc < K;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      float4 a = r.a[i];
      if (LN)
        a = make_float4((a.x - mu[i]) * rs[i] * rg.x + rb.x, (a.y - mu[i]) * rs[i] * rg.y + rb.y,
                        (a.z - mu[i]) * rs[i] * rg.z + rb.z, (a.w - mu[i]) * rs[i] * rg.w + rb.w);
      if (MUL) {
        const float4 q = r.m[MUL ? i : 0];
        a = make_float4(a.x * q.x, a.y * q.y, a.z * q.z, a.w * q.w);
      }
      *(float4*)(sa + buf * SA + (pr + RA * i) * kPA + pc) = WHOLE ? a : keep_if(a, kok);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if (LAYOUT == MPL_W_IN_OUT)
        *(float4*)(sw + buf * SW + (wr + 16 * i) * kPW + wc) = WHOLE ? r.w[i] : keep_if(r.w[i], k0 + wr + 16 * i < K);
      else
        *(float4*)(sw + buf * SW + (wr + RA * i) * kPA + wc) = WHOLE ? r.w[i] : keep_if(r.w[i], kok);
    }
  };

  const int col = lane & 31, h = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  const float* pa = sa + (32 * wm + col) * kPA + 4 * h;
  const float* pw = LAYOUT == MPL_W_IN_OUT ? sw + 4 * h * kPW + 32 * wn + col : sw + (32 * wn + col) * kPA + 4 * h;
  f32x16 acc = f32x16{};
  constexpr int G = kKC / 8;  // groups of four MFMAs a chunk
  float4 oa[G], ob[G];        // the chunk's operands
  auto operands = [&](int g, int buf) __attribute__((always_inline)) {
    const float *ca = pa + buf * SA + 8 * g, *cw = pw + buf * SW;
    oa[g] = *(const float4*)ca;
    if (LAYOUT == MPL_W_IN_OUT)
      ob[g] = make_float4(cw[(8 * g + 0) * kPW], cw[(8 * g + 1) * kPW], cw[(8 * g + 2) * kPW], cw[(8 * g + 3) * kPW]);
    else
      ob[g] = *(const float4*)(cw + 8 * g);
  };
  auto mfma4 = [&](float4 a, float4 b) __attribute__((always_inline)) {
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, acc, 0, 0, 0);
  };
  // One chunk, its operands in registers: the MFMAs of all groups but the
  // last with the next chunk's way into the other buffer between them (r, and
  // with FETCH the loads of the chunk two later into r); then the next
  // chunk's operands are on their way while the last group runs.
  auto chunk = [&](Pieces& r, int k0, int buf, auto FETCH, auto WHOLE) __attribute__((always_inline)) {
    stage(r, k0 + kKC, buf ^ 1, WHOLE);
    if (FETCH) fetch(r, k0 + 3 * kKC, WHOLE);
    if (LN) fetch_ln(k0 + 2 * kKC);
#pragma unroll
    for (int g = 0; g < G - 1; ++g) mfma4(oa[g], ob[g]);
    // MFMAs wait for one another, and what follows one in program order
    // waits with it: a few of the other instructions after each
#pragma unroll
    for (int g = 0; g < 4 * (G - 1); ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                    // MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, LN ? 8 : 5, 0);           // VALU
      if (g & 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);         // LDS write
      if (g & 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);         // load
    }
    __syncthreads();
    const float4 la = oa[G - 1], lb = ob[G - 1];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; ++g) operands(g, buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    mfma4(la, lb);
    __builtin_amdgcn_sched_barrier(0);
  };
  stage(set0, 0, 0, No{});
  fetch(set0, 2 * kKC, No{});
  if (LN) fetch_ln(kKC);
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g) operands(g, 0);
  int k0 = 0;
  for (; k0 + 5 * kKC <= K; k0 += 2 * kKC) {  // what is fetched here lies below K
    chunk(set1, k0, 0, Yes{}, Whole{});
    chunk(set0, k0 + kKC, 1, Yes{}, Whole{});
    if (LN) continue;
    at_k += 2 * kKC;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      xp[i] += 2 * kKC;
      if (MUL) mp[MUL ? i : 0] += 2 * kKC;
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) wp[i] += LAYOUT == MPL_W_IN_OUT ? (int64_t)2 * kKC * L.N : (int64_t)2 * kKC;
  }
  // up to five chunks left
  if (k0 + kKC < K) chunk(set1, k0, 0, Yes{}, No{});
  if (k0 + 2 * kKC < K) chunk(set0, k0 + kKC, 1, Yes{}, No{});
  if (k0 + 3 * kKC < K) chunk(set1, k0 + 2 * kKC, 0, No{}, No{});
  if (k0 + 4 * kKC < K) chunk(set0, k0 + 3 * kKC, 1, No{}, No{});
#pragma unroll
  for (int g = 0; g < G; ++g) mfma4(oa[g], ob[g]);

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
  DenseArgs a{x, x_mul, ln_scale, ln_bias, residual, rows, K, count, 0, ln_eps, {}};
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
  a.tiles = (uint32_t)tiles;
  const int64_t groups = tiles * cdiv(rows, kTM);
  MPL_REQUIRE(groups < ((int64_t)1 << 31), MPL_EUNSUPPORTED, "mpl_dense_layers: too many tiles");
  const dim3 grid((unsigned)groups);
  if (weight_layout == MPL_W_OUT_IN) launch_dense<MPL_W_OUT_IN>(a, grid, (hipStream_t)stream);
  else launch_dense<MPL_W_IN_OUT>(a, grid, (hipStream_t)stream);
  return check_launch("mpl_dense_layers");
}
