// Minibatch index draw and row gather (DeviceNumpyDataLoader.get_random_data,
// data/numpy_loader.py:128-141, and tree_index, data/core.py:642-660).
#include <type_traits>

#include "sgmc_common.h"
#include "sgmc_device.h"

namespace sgmc {

constexpr int kNT = 256;

// (dkey_out, sub) = split(dkey_in); idx = randint(sub, (n,), 0, N).
__global__ void __launch_bounds__(kNT) draw_batch_kernel(const uint32_t* __restrict__ dkey_in,
                                                         uint32_t* __restrict__ dkey_out,
                                                         int32_t* __restrict__ idx, uint32_t n,
                                                         uint32_t span, uint32_t mult,
                                                         uint32_t magic) {
  Key next, sub, k1, k2;
  split2(load_key(dkey_in), next, sub);
  split2(sub, k1, k2);
  const uint32_t m = (n + 1) >> 1;
  const uint32_t j = blockIdx.x * kNT + threadIdx.x;
  if (j < m) {
    uint32_t h0, h1, l0, l1;
    bits_pair(k1, n, j, h0, h1);
    bits_pair(k2, n, j, l0, l1);
    idx[j] = (int32_t)randint_offset(h0, l0, span, mult, magic);
    if (j + m < n) idx[j + m] = (int32_t)randint_offset(h1, l1, span, mult, magic);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) store_key(dkey_out, next);
}

// Rows of `row_vecs` elements T gathered as one flat run of n row_vecs elements, kFlat per
// thread in flight: a wavefront per row leaves lanes idle in the row's last load (19 of 64
// carry data at 76 16-byte elements) and one lane of 64 working on 4-byte rows. Per gather, n = 40001
// rows of 1216 bytes 17.3 -> 16.2 us, of 4 bytes 4.7 -> 2.4; n = 60000 of 48 bytes 6.8 -> 2.7.
// Rows whose index lies outside the source are left as they are.
template <class T, int kFlat>
__global__ void __launch_bounds__(kNT) gather_flat_kernel(const T* __restrict__ src,
                                                          const int32_t* __restrict__ idx,
                                                          T* __restrict__ dst, uint32_t total,
                                                          uint32_t row_vecs, uint32_t magic,
                                                          int64_t src_stride_vecs,
                                                          int64_t src_rows) {
  const uint32_t f0 = blockIdx.x * (uint32_t)(kFlat * kNT) + threadIdx.x;
  T v[kFlat];
  bool ok[kFlat];
#pragma unroll
  for (int u = 0; u < kFlat; ++u) {
    const uint32_t f = f0 + u * kNT;
    ok[u] = f < total;
    const uint32_t g = ok[u] ? f : total - 1;
    // row = g / row_vecs: umulhi(g, floor(2^32 / row_vecs)) is it or one less
    uint32_t row = row_vecs == 1 ? g : __umulhi(g, magic);
    if (g - row * row_vecs >= row_vecs) ++row;
    const int64_t r = (int64_t)idx[row];
    ok[u] = ok[u] && (uint64_t)r < (uint64_t)src_rows;
    v[u] = src[(ok[u] ? r : 0) * src_stride_vecs + (g - row * row_vecs)];
  }
#pragma unroll
  for (int u = 0; u < kFlat; ++u)
    if (ok[u]) dst[f0 + u * kNT] = v[u];
}

// One wavefront per row, for rows of any byte length and gathers of 2^31 elements or more.
template <class T>
__global__ void __launch_bounds__(kNT) gather_row_kernel(const T* __restrict__ src,
                                                         const int32_t* __restrict__ idx,
                                                         T* __restrict__ dst, int n,
                                                         int64_t row_vecs,
                                                         int64_t src_stride_vecs,
                                                         int64_t src_rows) {
  const int row = blockIdx.x * (kNT / kWave) + threadIdx.x / kWave;
  if (row >= n) return;
  if ((uint64_t)(int64_t)idx[row] >= (uint64_t)src_rows) return;
  const int lane = threadIdx.x & (kWave - 1);
  const T* s = src + (int64_t)idx[row] * src_stride_vecs;
  T* d = dst + (int64_t)row * row_vecs;
  for (int64_t c = lane; c < row_vecs; c += kWave) d[c] = s[c];
}

template <class T>
void launch_gather(const void* src, int64_t src_rows, const int32_t* idx, void* dst, int n,
                   int64_t row_bytes, int64_t src_stride_bytes, hipStream_t s) {
  const int64_t vecs = row_bytes / sizeof(T), stride = src_stride_bytes / sizeof(T);
  const int64_t total = (int64_t)n * vecs;
  if (src_rows >= 1 && total < (int64_t(1) << 31)) {
    // one element per thread until that fills the device (small gathers are one latency)
    const auto go = [&](auto per) {
      constexpr int kFlat = decltype(per)::value;
      const int64_t blocks = (total + kFlat * kNT - 1) / (kFlat * kNT);
      hipLaunchKernelGGL((gather_flat_kernel<T, kFlat>), dim3((unsigned)blocks), dim3(kNT), 0, s,
                         (const T*)src, idx, (T*)dst, (uint32_t)total, (uint32_t)vecs,
                         randint_magic((uint32_t)vecs), stride, src_rows);
    };
    if (total <= 1 << 19) go(std::integral_constant<int, 1>{});
    else go(std::integral_constant<int, 4>{});
  } else {
    const int rows_per_block = kNT / kWave;
    hipLaunchKernelGGL(gather_row_kernel<T>, dim3((n + rows_per_block - 1) / rows_per_block),
                       dim3(kNT), 0, s, (const T*)src, idx, (T*)dst, n, vecs, stride, src_rows);
  }
}

}  // namespace sgmc

using namespace sgmc;

extern "C" {

int sgmc_draw_batch(const uint32_t* dkey_in, uint32_t* dkey_out, int32_t* idx, int n,
                    int64_t N, void* stream) {
  SGMC_REQUIRE(dkey_in && dkey_out && idx, SGMC_E_ARG, "sgmc_draw_batch: null pointer");
  SGMC_REQUIRE(dkey_in != dkey_out, SGMC_E_ARG,
               "sgmc_draw_batch: dkey_in and dkey_out must not alias");
  SGMC_REQUIRE(n >= 1, SGMC_E_ARG, "sgmc_draw_batch: batch size must be positive, got %d", n);
  SGMC_REQUIRE(N >= 1 && N <= 2147483647LL, SGMC_E_ARG,
               "sgmc_draw_batch: observation count %lld out of int32 range", (long long)N);
  const uint32_t span = (uint32_t)N;
  const uint32_t m = ((uint32_t)n + 1) >> 1;
  hipLaunchKernelGGL(draw_batch_kernel, dim3((m + kNT - 1) / kNT), dim3(kNT), 0,
                     as_stream(stream), dkey_in, dkey_out, idx, (uint32_t)n, span,
                     randint_mult(span), randint_magic(span));
  return check_launch("sgmc_draw_batch");
}

int sgmc_gather_rows(const void* src, int64_t src_rows, const int32_t* idx, void* dst, int n,
                     int64_t row_bytes, int64_t src_stride_bytes, void* stream) {
  SGMC_REQUIRE(src && idx && dst, SGMC_E_ARG, "sgmc_gather_rows: null pointer");
  SGMC_REQUIRE(n >= 0 && row_bytes >= 0 && src_stride_bytes >= row_bytes, SGMC_E_ARG,
               "sgmc_gather_rows: bad shape");
  if (n == 0 || row_bytes == 0) return SGMC_OK;
  const uint64_t all = (uint64_t)(uintptr_t)src | (uint64_t)(uintptr_t)dst |
                       (uint64_t)row_bytes | (uint64_t)src_stride_bytes;
  hipStream_t s = as_stream(stream);
  if (all % 16 == 0)
    launch_gather<uint4>(src, src_rows, idx, dst, n, row_bytes, src_stride_bytes, s);
  else if (all % 4 == 0)
    launch_gather<uint32_t>(src, src_rows, idx, dst, n, row_bytes, src_stride_bytes, s);
  else
    launch_gather<uint8_t>(src, src_rows, idx, dst, n, row_bytes, src_stride_bytes, s);
  return check_launch("sgmc_gather_rows");
}

}  // extern "C"
