// Stage 1 for key ranges of a few blocks a wave: cosine scoring on MFMA and
// the exact top-k by sorting in registers (memory.py:149-164, no noise).
//
// A workgroup is one wave: 32 queries of one codebook hc and one split of its
// keys.  Scoring is score_topk_kernel's (score_select.hip), bit for bit: each
// block of 32 keys is one chain of 32x32 MFMAs with the keys as the A operand,
// so lanes l and l + 32 hold 16 scores of query l % 32 each.  A lane turns its
// 16 scores of a block into keys (topk.h), sorts them (60 compare-exchanges)
// and merges them into its sorted list of the best KMAX (16 maxima and a
// bitonic merger); the lane pair's lists meet at the end.  No LDS, no
// thresholds, no candidate buffers and one scoring pass: the time does not
// depend on the scores.
//
// Bound: the VALU, about 1,850 cycles a block and wave (92 compare-exchanges
// of two double-precision instructions each), with the next block's MFMAs
// and key loads issued beside them (fp16).
//
// This file is compiled without IEEE mode and NaN handling of min / max (no
// canonicalisation of the keys, which the compiler would otherwise add to
// every value it cannot trace: +28% double-precision instructions).  NaN scores
// are turned into -FLT_MAX, by their bits, before they become keys (no cosine
// is that small; the output takes it for "none"), so no key is a NaN.
#include <float.h>

#include "score_stage1.h"
#include "topk.h"

namespace mpl {

template <typename T, int HP, int KMAX>
__global__ __launch_bounds__(kWave, 2) void score_sort_kernel(ScoreParams p) {
  constexpr int VPL = KeyPack<T>::vectors_per_lane(HP);
  constexpr int OPV = KeyPack<T>::kOpsPerVec;
  constexpr int NCH = VPL * OPV;
  constexpr int TILE = VPL * kWave;  // uint4 per key block
  typedef typename Mfma<T>::Op Op;

  const int lane = threadIdx.x;
  const int par = lane >> 5;
  // wave-uniform, but the divisions leave them in vector registers
  const int hc = __builtin_amdgcn_readfirstlane(blockIdx.x % p.HC);
  const int split = __builtin_amdgcn_readfirstlane((blockIdx.x / p.HC) % p.splits);
  const int qb = __builtin_amdgcn_readfirstlane(blockIdx.x / (p.HC * p.splits));
  const int64_t my_q = (int64_t)qb * kQueriesPerWave + (lane & 31);
  const bool valid = my_q < p.M;
  const int b_begin = split * p.blk_per_split;
  const int b_end = min(p.nblk, b_begin + p.blk_per_split);  // the plan leaves no split empty

  const uint4* kbase = p.packed + (int64_t)hc * p.nblk * TILE + lane;
  uint4 u[VPL];  // the lane's A operand of the block scored next
#pragma unroll
  for (int v = 0; v < VPL; ++v) u[v] = kbase[(int64_t)b_begin * TILE + v * kWave];
  __builtin_amdgcn_sched_barrier(0);  // keys and queries in one memory round trip
  Op qop[NCH];
  float ql;
  query_operand<T, NCH>(p, hc, my_q, valid, lane, split == 0, qop, ql);

  // The scores of the block in u; u takes block nb (clamped to the split).
  auto score = [&](int nb) __attribute__((always_inline)) {
    const uint4* src = kbase + (int64_t)min(nb, b_end - 1) * TILE;
    f32x16 x = f32x16{};
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
#pragma unroll
      for (int e = 0; e < OPV; ++e) x = Mfma<T>::mma(Mfma<T>::from_vec(u[v], e), qop[v * OPV + e], x);
      u[v] = src[v * kWave];
    }
    return x;
  };
  // NaN scores of a block become -FLT_MAX, by integer operations on their
  // bits: the compiler takes every float of this file for a number.  Cosines
  // are below 2, so one test of the bits of all 16 (bit 30: 2 and above, inf
  // and NaN) decides for the wave whether any has to be looked at.
  auto drop_nans = [&](f32x16& x) __attribute__((always_inline)) {
    asm("" : "+v"(x));  // no assumption about the MFMAs' results passes here
    uint32_t any = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) any |= __float_as_uint(x[r]);
    if (__ballot((any & 0x40000000u) != 0) != 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t u = __float_as_uint(x[r]);
        x[r] = __uint_as_float((u & 0x7FFFFFFFu) > 0x7F800000u ? 0xFF7FFFFFu : u);
      }
    }
  };
  // The lane's keys of block b, sorted.  MFMA sums start at +0, so a score is
  // -0 only where its exact value is negative and underflows; below a negative
  // score the index is stored uncomplemented (topk.h).
  auto sorted_keys = [&](int b, const f32x16& x, Key (&c)[16]) __attribute__((always_inline)) {
    const uint32_t nidx = ~(uint32_t)(b * 32 + 4 * par);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t hi = __float_as_uint(x[r]);
      c[r] = key_of(hi, (nidx - (uint32_t)(8 * (r >> 2) + (r & 3))) ^ (uint32_t)((int)hi >> 31));
    }
    if (b * 32 + 32 > p.n) {  // wave-uniform: only the last block can hold padded keys
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (b * 32 + 8 * (r >> 2) + 4 * par + (r & 3) >= p.n) c[r] = kNoKey;
    }
    sort16(c);
  };

  TopList<KMAX, false> top;
  top.init();
  Key c[16];
  f32x16 x = score(b_begin + 1);
  if constexpr (sizeof(T) == 2) {
    // the next block's MFMAs beside this block's sort; past the end they
    // score the last block again and nobody reads them
    for (int b = b_begin; b < b_end; ++b) {
      drop_nans(x);
      const f32x16 y = score(b + 2);
      sorted_keys(b, x, c);
      if (b == b_begin) {  // wave-uniform: the list is empty
#pragma unroll
        for (int i = 0; i < 16; ++i) top.key[i] = c[i];
      } else {
        top.template merge<16>(c, nullptr);
      }
      x = y;
    }
  } else {
    // fp32 MFMAs take longer than the sort: none is issued for nothing
    for (int b = b_begin; b < b_end; ++b) {
      if (b > b_begin) x = score(b + 1);
      drop_nans(x);
      sorted_keys(b, x, c);
      if (b == b_begin) {
#pragma unroll
        for (int i = 0; i < 16; ++i) top.key[i] = c[i];
      } else {
        top.template merge<16>(c, nullptr);
      }
    }
  }

  // The partner lane's list (keys of the other parity) joins this lane's:
  // both lanes of a query end with its best KMAX, and each writes half.
  {
    Key other[KMAX];
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      float lo = __uint_as_float(key_lo(top.key[j])), lo2 = lo;
      float hi = __uint_as_float(key_hi(top.key[j])), hi2 = hi;
      half_swap(lo, lo2);
      half_swap(hi, hi2);
      other[j] = key_of(__float_as_uint(par ? hi : hi2), __float_as_uint(par ? lo : lo2));
    }
    top.template merge<KMAX>(other, nullptr);
  }
  if (!valid) return;
  const float Tv = *p.T;
  constexpr int W = KMAX / 2;
  const int r0 = par * W;
  float cl[W];
  int id[W];
#pragma unroll
  for (int r = 0; r < W; ++r) {
    const Key kk = par ? top.key[W + r] : top.key[r];
    const float s = key_score(kk);
    const bool some = s > -FLT_MAX;  // else no key, or one of a NaN
    float clean = s * Tv;
    clean *= ql;  // ql == 1 without query_scale
    cl[r] = some ? clean : -INFINITY;
    id[r] = some ? key_index(kk) : -1;
  }
  const int64_t o = (((int64_t)split * p.M + my_q) * p.HC + hc) * p.k + r0;
  if (p.k == KMAX && ((uintptr_t)(p.out_clean + o) & 15) == 0 && ((uintptr_t)(p.out_idx + o) & 15) == 0) {
#pragma unroll
    for (int r = 0; r < W; r += 4) {
      *(float4*)(p.out_clean + o + r) = make_float4(cl[r], cl[r + 1], cl[r + 2], cl[r + 3]);
      *(int4*)(p.out_idx + o + r) = make_int4(id[r], id[r + 1], id[r + 2], id[r + 3]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < W; ++r) {
      if (r0 + r < p.k) {
        p.out_clean[o + r] = cl[r];
        p.out_idx[o + r] = id[r];
      }
    }
  }
}

template <typename T, int HP>
static void launch_kmax(const ScoreParams& sp, int kmax, unsigned grid, hipStream_t s) {
  if (kmax == 16) score_sort_kernel<T, HP, 16><<<grid, kWave, 0, s>>>(sp);
  else score_sort_kernel<T, HP, 32><<<grid, kWave, 0, s>>>(sp);
}

int launch_score_sort(const ScoreParams& sp, int score_dtype, int HP, int kmax, hipStream_t s) {
  const unsigned grid = (unsigned)(cdiv(sp.M, kQueriesPerWave) * sp.splits * sp.HC);
  if (score_dtype == MPL_F16) {
    switch (HP) {
      case 16: launch_kmax<_Float16, 16>(sp, kmax, grid, s); break;
      case 32: launch_kmax<_Float16, 32>(sp, kmax, grid, s); break;
      case 64: launch_kmax<_Float16, 64>(sp, kmax, grid, s); break;
      case 128: launch_kmax<_Float16, 128>(sp, kmax, grid, s); break;
      default: return MPL_EUNSUPPORTED;
    }
  } else {
    switch (HP) {
      case 8: launch_kmax<float, 8>(sp, kmax, grid, s); break;
      case 16: launch_kmax<float, 16>(sp, kmax, grid, s); break;
      case 32: launch_kmax<float, 32>(sp, kmax, grid, s); break;
      case 64: launch_kmax<float, 64>(sp, kmax, grid, s); break;
      case 128: launch_kmax<float, 128>(sp, kmax, grid, s); break;
      default: return MPL_EUNSUPPORTED;
    }
  }
  return MPL_OK;
}

}  // namespace mpl
