// Value read: out[m] = sum over the H*k fetched rows of w * values[slot]
// (memory.py:179-193), without materialising the fetched rows.  One wave per
// token; the row sum itself is Wsum (wsum.h), shared with the fused stage-2
// kernel of score_select.hip.
#include "common.h"
#include "wsum.h"

namespace mpl {

constexpr int kGatherThreads = 256;

template <typename V, int VR, bool NT, bool WHOLE>
__global__ __launch_bounds__(kGatherThreads) void gather_wsum_kernel(
    const V* __restrict__ values, int64_t N, const int32_t* __restrict__ slots,
    const float* __restrict__ weights, int64_t M, int R, int shuffle, float* __restrict__ out) {
  const int64_t m = (int64_t)blockIdx.x * (kGatherThreads / kWave) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (m >= M) return;
  Wsum<V, VR, 32, NT> acc;
  const uint4* base = (const uint4*)values;
  for (int r0 = 0; r0 < R; r0 += kWave) {
    const int rr = r0 + lane;
    const bool in = rr < R;
    int sl = slots[m * R + (in ? rr : 0)];  // unconditional (clamped) loads
    float ww = weights[m * R + (in ? rr : 0)];
    if (shuffle) sl = (int)(((int64_t)sl + N / 2 + 1) % N);
    sl = in ? (int)min(max((int64_t)sl, (int64_t)0), N - 1) : 0;  // out-of-range ids read the nearest row
    ww = in ? ww : 0.f;
    acc.template add_chunk<WHOLE>(base, sl, ww, min(kWave, R - r0), lane);
  }
  acc.store(out + m * (int64_t)(VR * Vec16<V>::kElems), lane);
}

// Rows of any other number of 16-byte vectors up to 64 (WsumAny).
template <typename V, bool NT>
__global__ __launch_bounds__(kGatherThreads) void gather_wsum_any(
    const V* __restrict__ values, int64_t N, int VR, const int32_t* __restrict__ slots,
    const float* __restrict__ weights, int64_t M, int R, int shuffle, float* __restrict__ out) {
  const int64_t m = (int64_t)blockIdx.x * (kGatherThreads / kWave) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (m >= M) return;
  WsumAny<V, NT> acc(VR, lane);
  for (int r0 = 0; r0 < R; r0 += kWave) {
    const int rr = r0 + lane;
    const bool in = rr < R;
    int sl = slots[m * R + (in ? rr : 0)];  // unconditional (clamped) loads
    float ww = weights[m * R + (in ? rr : 0)];
    if (shuffle) sl = (int)(((int64_t)sl + N / 2 + 1) % N);
    sl = in ? (int)min(max((int64_t)sl, (int64_t)0), N - 1) : 0;  // out-of-range ids read the nearest row
    ww = in ? ww : 0.f;
    acc.add_chunk((const uint4*)values, sl, ww, min(kWave, R - r0));
  }
  acc.store(out + m * (int64_t)VR * WsumAny<V, NT>::VE, lane);
}

// Any d: one thread per (token, column).
template <typename V>
__global__ __launch_bounds__(256) void gather_wsum_generic(const V* __restrict__ values, int64_t N, int d,
                                                          const int32_t* __restrict__ slots,
                                                          const float* __restrict__ weights, int64_t M,
                                                          int R, int shuffle, float* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M * d) return;
  const int64_t m = t / d;
  const int j = (int)(t % d);
  float acc = 0.f;
  for (int r = 0; r < R; ++r) {
    int64_t s = slots[m * R + r];
    if (shuffle) s = (s + N / 2 + 1) % N;
    s = s < 0 ? 0 : (s >= N ? N - 1 : s);
    acc = fmaf(weights[m * R + r], (float)values[s * d + j], acc);
  }
  out[t] = acc;
}

template <typename V>
static int gather_impl(const V* values, int64_t N, int d, const int32_t* slots, const float* w, int64_t M,
                       int R, int shuffle, float* out, hipStream_t s) {
  const int64_t bytes = (int64_t)d * sizeof(V);
  const unsigned blocks = (unsigned)cdiv(M, kGatherThreads / kWave);
  if (bytes % 16 == 0 && ((uintptr_t)values % 16) == 0 && ((uintptr_t)out % 16) == 0) {
    const int VR = (int)(bytes / 16);
    const bool nt = N * bytes > kStreamTableBytes;
    switch (VR) {
#define MPL_GK(vr, NT, WHOLE) \
  gather_wsum_kernel<V, vr, NT, WHOLE><<<blocks, kGatherThreads, 0, s>>>(values, N, slots, w, M, R, shuffle, out)
#define MPL_G(vr)                                   \
  case vr:                                          \
    if (R % kWave == 0) {                           \
      if (nt) MPL_GK(vr, true, true);               \
      else MPL_GK(vr, false, true);                 \
    } else {                                        \
      if (nt) MPL_GK(vr, true, false);              \
      else MPL_GK(vr, false, false);                \
    }                                               \
    return check_launch("mpl_gather_wsum");
      MPL_G(1) MPL_G(2) MPL_G(4) MPL_G(8) MPL_G(16) MPL_G(32) MPL_G(64) MPL_G(128) MPL_G(256)
#undef MPL_G
#undef MPL_GK
      default: break;
    }
    if (VR <= kWave) {
      if (nt) gather_wsum_any<V, true><<<blocks, kGatherThreads, 0, s>>>(values, N, VR, slots, w, M, R, shuffle, out);
      else gather_wsum_any<V, false><<<blocks, kGatherThreads, 0, s>>>(values, N, VR, slots, w, M, R, shuffle, out);
      return check_launch("mpl_gather_wsum");
    }
  }
  gather_wsum_generic<V><<<(unsigned)cdiv(M * d, 256), 256, 0, s>>>(values, N, d, slots, w, M, R, shuffle, out);
  return check_launch("mpl_gather_wsum(generic)");
}

// Row copy for the host tier: out[i] = table[clamp(idx[i])] for i < rows,
// rows = min(count, *count_dev) (count_dev may be null).  The table may be
// device memory or pinned host memory mapped for the device, in which case
// every 16-byte vector crosses the bus once; kUnroll vectors per thread are
// loaded before any is stored, so several reads are in flight per lane.
constexpr int kRowCopyUnroll = 4;

template <int W>
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint32_t* __restrict__ table, int64_t N, int wpr,
                                                          const int32_t* __restrict__ idx, int64_t count,
                                                          const int32_t* __restrict__ count_dev,
                                                          uint32_t* __restrict__ out) {
  // W 32-bit words per access (4: 16-byte vectors); wpr accesses per row
  typedef uint32_t Acc __attribute__((ext_vector_type(W)));
  const int64_t rows = count_dev != nullptr ? min(count, (int64_t)*count_dev) : count;
  const int64_t total = rows * wpr;
  const int64_t stride = (int64_t)gridDim.x * 256 * kRowCopyUnroll;
  for (int64_t t0 = (int64_t)blockIdx.x * 256 * kRowCopyUnroll + threadIdx.x; t0 < total; t0 += stride) {
    Acc v[kRowCopyUnroll];
    int64_t dst[kRowCopyUnroll];
#pragma unroll
    for (int u = 0; u < kRowCopyUnroll; ++u) {
      const int64_t t = t0 + (int64_t)u * 256;
      const bool ok = t < total;
      const int64_t r = ok ? t / wpr : 0;
      const int c = ok ? (int)(t - r * wpr) : 0;
      int64_t sl = idx[r];
      sl = sl < 0 ? 0 : (sl >= N ? N - 1 : sl);
      v[u] = ((const Acc*)table)[sl * wpr + c];
      dst[u] = ok ? t : -1;
    }
#pragma unroll
    for (int u = 0; u < kRowCopyUnroll; ++u)
      if (dst[u] >= 0) ((Acc*)out)[dst[u]] = v[u];
  }
}

// out[idx[i]] = rows[i] for the first min(count, *count_dev) entries whose
// index lies in [0, N): a wave a row, W words a lane.  Bound: HBM, each row
// read and written once.  As the table's dense gradient (16,384 rows of 1 KB)
// it replaces an id conversion, a scatter through 64-bit ids and the zeroing
// of the merge's padding: with its merge (8,192 tokens, 16,384 rows) 122.0 us
// for 141.5, this kernel 7.1 of them.
template <int W>
__global__ __launch_bounds__(256) void scatter_rows_kernel(const uint32_t* __restrict__ rows,
                                                           const int32_t* __restrict__ idx, int64_t count,
                                                           const int32_t* __restrict__ count_dev, int64_t N, int wpr,
                                                           uint32_t* __restrict__ out) {
  typedef uint32_t Acc __attribute__((ext_vector_type(W)));
  const int64_t n = count_dev != nullptr ? min(count, (int64_t)*count_dev) : count;
  const int lane = threadIdx.x & 63;
  for (int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); i < n; i += (int64_t)gridDim.x * 4) {
    const int64_t to = idx[i];
    if (to < 0 || to >= N) continue;
    for (int c = lane; c < wpr; c += kWave) ((Acc*)out)[to * wpr + c] = ((const Acc*)rows)[i * wpr + c];
  }
}

// Copies of up to kMaxCopies arrays of 32-bit words in one launch: a block
// copies kCopyWords of one of them, 16 bytes a lane where both ends are
// aligned.  Bound: memory (24 MB moved for two layers' fetches, 7.3 us, where
// three library concatenations take 19.7).  One vector a lane: four in a local
// array went through 16 KB of LDS a block (20.1 us).
constexpr int kMaxCopies = 12;
constexpr int kCopyWords = 256 * 4;
struct CopyArgs {
  const uint32_t* src[kMaxCopies];
  uint32_t* dst[kMaxCopies];
  int64_t words[kMaxCopies];
  uint32_t block0[kMaxCopies];  // the first block of each
  int count;
};

__global__ __launch_bounds__(256) void copy_arrays_kernel(CopyArgs p) {
  // the block's array, by selects at constant places of the arguments
  const uint32_t* src = p.src[0];
  uint32_t* dst = p.dst[0];
  int64_t words = p.words[0];
  uint32_t b0 = 0;
#pragma unroll
  for (int i = 1; i < kMaxCopies; ++i) {
    const bool past = i < p.count && blockIdx.x >= p.block0[i];
    src = past ? p.src[i] : src;
    dst = past ? p.dst[i] : dst;
    words = past ? p.words[i] : words;
    b0 = past ? p.block0[i] : b0;
  }
  const int64_t w0 = (int64_t)(blockIdx.x - b0) * kCopyWords, end = min(w0 + kCopyWords, words);
  if (((((uintptr_t)src) | ((uintptr_t)dst)) & 15) == 0) {
    const int64_t at = w0 + 4 * threadIdx.x;
    if (at + 4 <= end) *(uint4*)(dst + at) = *(const uint4*)(src + at);
    const int64_t rest = w0 + (end - w0) / 4 * 4 + threadIdx.x;  // the last 0 to 3 words
    if (rest < end) dst[rest] = src[rest];
  } else {
    for (int64_t w = w0 + threadIdx.x; w < end; w += 256) dst[w] = src[w];
  }
}

}  // namespace mpl

using namespace mpl;

extern "C" int mpl_scatter_rows(const float* rows, const int32_t* idx, int64_t count, const int32_t* count_dev, int d,
                                int64_t N, float* out, void* stream) {
  clear_error();
  MPL_REQUIRE(N > 0 && d > 0 && count >= 0, MPL_EINVAL, "mpl_scatter_rows: bad sizes N=%lld d=%d count=%lld",
              (long long)N, d, (long long)count);
  if (count == 0) return MPL_OK;
  MPL_REQUIRE(rows && idx && out, MPL_EINVAL, "mpl_scatter_rows: null buffer");
  hipStream_t s = (hipStream_t)stream;
  const bool vec = d % 4 == 0 && ((uintptr_t)rows % 16) == 0 && ((uintptr_t)out % 16) == 0;
  const unsigned blocks = (unsigned)(cdiv(count, 4) < 8192 ? cdiv(count, 4) : 8192);
  if (vec)
    scatter_rows_kernel<4><<<blocks, 256, 0, s>>>((const uint32_t*)rows, idx, count, count_dev, N, d / 4, (uint32_t*)out);
  else
    scatter_rows_kernel<1><<<blocks, 256, 0, s>>>((const uint32_t*)rows, idx, count, count_dev, N, d, (uint32_t*)out);
  return check_launch("mpl_scatter_rows");
}

extern "C" int mpl_copy_arrays(const void* srcs, const void* dsts, const void* words, int count, void* stream) {
  clear_error();
  MPL_REQUIRE(count >= 0 && count <= kMaxCopies, MPL_EINVAL, "mpl_copy_arrays: count=%d (at most %d)", count, kMaxCopies);
  if (count == 0) return MPL_OK;
  MPL_REQUIRE(srcs && dsts && words, MPL_EINVAL, "mpl_copy_arrays: null table");
  CopyArgs a{};
  int64_t blocks = 0;
  for (int i = 0; i < count; ++i) {
    const int64_t n = ((const int64_t*)words)[i];
    MPL_REQUIRE(n >= 0, MPL_EINVAL, "mpl_copy_arrays: array %d has %lld words", i, (long long)n);
    if (n == 0) continue;
    const int at = a.count++;
    a.src[at] = ((const uint32_t* const*)srcs)[i];
    a.dst[at] = ((uint32_t* const*)dsts)[i];
    a.words[at] = n;
    a.block0[at] = (uint32_t)blocks;
    MPL_REQUIRE(a.src[at] && a.dst[at], MPL_EINVAL, "mpl_copy_arrays: array %d: null buffer", i);
    blocks += cdiv(n, kCopyWords);
    MPL_REQUIRE(blocks < ((int64_t)1 << 31), MPL_EUNSUPPORTED, "mpl_copy_arrays: arrays too large");
  }
  if (blocks == 0) return MPL_OK;
  copy_arrays_kernel<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(a);
  return check_launch("mpl_copy_arrays");
}

extern "C" int mpl_gather_rows(const void* table, int dtype, int64_t N, int d, const int32_t* idx, int64_t count,
                               const int32_t* count_dev, void* out, void* stream) {
  clear_error();
  MPL_REQUIRE(N > 0 && d > 0 && count >= 0, MPL_EINVAL, "mpl_gather_rows: bad sizes N=%lld d=%d count=%lld",
              (long long)N, d, (long long)count);
  MPL_REQUIRE(dtype == MPL_F16 || dtype == MPL_F32, MPL_EINVAL, "mpl_gather_rows: dtype must be MPL_F16 or MPL_F32");
  if (count == 0) return MPL_OK;
  MPL_REQUIRE(table && idx && out, MPL_EINVAL, "mpl_gather_rows: null buffer");
  const int64_t row_bytes = (int64_t)d * (dtype == MPL_F16 ? 2 : 4);
  MPL_REQUIRE(row_bytes % 4 == 0, MPL_EUNSUPPORTED, "mpl_gather_rows: rows of %lld bytes (need a multiple of 4)",
              (long long)row_bytes);
  hipStream_t s = (hipStream_t)stream;
  const bool vec = row_bytes % 16 == 0 && ((uintptr_t)table % 16) == 0 && ((uintptr_t)out % 16) == 0;
  const int wpr = (int)(vec ? row_bytes / 16 : row_bytes / 4);
  const int64_t work = cdiv(count * wpr, 256 * kRowCopyUnroll);
  const unsigned blocks = (unsigned)(work < 4096 ? (work > 0 ? work : 1) : 4096);
  if (vec)
    gather_rows_kernel<4><<<blocks, 256, 0, s>>>((const uint32_t*)table, N, wpr, idx, count, count_dev,
                                                 (uint32_t*)out);
  else
    gather_rows_kernel<1><<<blocks, 256, 0, s>>>((const uint32_t*)table, N, wpr, idx, count, count_dev,
                                                 (uint32_t*)out);
  return check_launch("mpl_gather_rows");
}

extern "C" int mpl_host_device_pointer(void* host_ptr, void** dev_ptr) {
  clear_error();
  MPL_REQUIRE(host_ptr && dev_ptr, MPL_EINVAL, "mpl_host_device_pointer: null argument");
  void* p = nullptr;
  const hipError_t e = hipHostGetDevicePointer(&p, host_ptr, 0);
  // the failed query is reported here; clear HIP's sticky per-thread error,
  // or the caller's next launch check would report it again
  if (e != hipSuccess) (void)hipGetLastError();
  MPL_REQUIRE(e == hipSuccess && p != nullptr, MPL_EINVAL,
              "mpl_host_device_pointer: %p is not pinned host memory mapped for the device (%s)", host_ptr,
              hipGetErrorString(e));
  *dev_ptr = p;
  return MPL_OK;
}

extern "C" int mpl_gather_wsum(const void* values, int values_dtype, int64_t N, int d, const int32_t* slots,
                               const float* weights, int64_t M, int R, int shuffle_reads, float* out,
                               void* stream) {
  clear_error();
  MPL_REQUIRE(N > 0 && d > 0 && M >= 0 && R > 0, MPL_EINVAL, "mpl_gather_wsum: bad sizes");
  if (M == 0) return MPL_OK;
  MPL_REQUIRE(values && slots && weights && out, MPL_EINVAL, "mpl_gather_wsum: null buffer");
  hipStream_t s = (hipStream_t)stream;
  if (values_dtype == MPL_F16)
    return gather_impl<_Float16>((const _Float16*)values, N, d, slots, weights, M, R, shuffle_reads, out, s);
  if (values_dtype == MPL_F32)
    return gather_impl<float>((const float*)values, N, d, slots, weights, M, R, shuffle_reads, out, s);
  set_error("mpl_gather_wsum: values_dtype must be MPL_F16 or MPL_F32");
  return MPL_EINVAL;
}
