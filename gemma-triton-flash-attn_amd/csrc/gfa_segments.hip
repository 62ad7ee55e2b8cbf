// Segment tables (include/gfa.h, seg_lo / seg_hi) from position ids or from a padding mask, one
// launch each. A model's attention layers each describe their batch this way, so the table is
// built once per layer call: built from framework operations it took up to twenty small launches
// (about 70 us of kernels for a (4, 1500) padding mask, and a device-to-host wait in the middle).
//
// One thread per token, 1024 per workgroup; every workgroup also scans its whole row for what
// lies outside its own 1024 tokens (the nearest segment start on either side, or the row's run
// of real tokens). That re-reads a row N / 1024 times from L2 (16 x 128 KB of position ids at
// N = 16384) and saves a second launch. Bound: latency, one row scan and one block scan.
#include "gfa_common.h"
#include "gfa_launch.h"

namespace gfa {

namespace {

constexpr int kTpb = 1024;
constexpr int kBatch = 8;  // tokens a thread has in flight while it scans a row
constexpr int kWaves = kTpb / 64;

// f(i) for this thread's tokens tid, tid + 1024, ... of a row of N: whole batches branch-free, so that
// their loads go out together (f's own branches aside), then the rest one by one. At N = 16384 the
// tables take 7.3 us, 8.9 us with a branch per token.
template <typename F>
__device__ __forceinline__ void scan_row(int N, int tid, F&& f) {
  int i = tid;
  for (; i + (kBatch - 1) * kTpb < N; i += kBatch * kTpb) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) f(i + j * kTpb);
  }
  for (; i < N; i += kTpb) f(i);
}

// Inclusive prefix max over the wave's lanes.
__device__ __forceinline__ int wave_scan_max(int x, int lane) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    const int y = __shfl_up(x, m);
    if (lane >= m) x = max(x, y);
  }
  return x;
}
// Inclusive suffix min over the wave's lanes.
__device__ __forceinline__ int wave_scan_min_rev(int x, int lane) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    const int y = __shfl_down(x, m);
    if (lane + m < 64) x = min(x, y);
  }
  return x;
}

}  // namespace

// Position ids: token i starts a sequence where its id is not the previous one plus one. lo = the
// last start at or before the token, hi = the first start after it (N past the last).
template <typename T>
__global__ __launch_bounds__(kTpb) void seg_positions_kernel(const T* pos, int64_t row_stride, int N, int* lo, int* hi) {
  __shared__ int w_last[kWaves], w_first[kWaves], w_before[kWaves], w_after[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* row = pos + (int64_t)blockIdx.y * row_stride;
  const int t0 = blockIdx.x * kTpb, t1 = min(N, t0 + kTpb);
  auto starts = [&](int i) {
    return (i == 0) | ((uint64_t)(int64_t)row[i] != (uint64_t)(int64_t)row[max(i - 1, 0)] + 1u);
  };

  int before = 0, after = N;  // nearest starts outside this workgroup's tokens (token 0 is one)
  auto outside = [&](int i) {
    const bool st = starts(i);
    before = max(before, st && i < t0 ? i : 0);
    after = min(after, st && i >= t1 ? i : N);
  };
  if (N > kTpb) scan_row(N, tid, outside);  // a row of one workgroup has nothing outside it
  const int i = t0 + tid;
  const bool st = i < N && starts(min(i, N - 1));
  const int last = wave_scan_max(st ? i : -1, lane);
  const int first = wave_scan_min_rev(st ? i : N, lane);
  before = wave_scan_max(before, lane);
  after = wave_scan_min_rev(after, lane);
  if (lane == 63) {
    w_last[wave] = last;
    w_before[wave] = before;
  }
  if (lane == 0) {
    w_first[wave] = first;
    w_after[wave] = after;
  }
  __syncthreads();
  int l = last;
  int f = __shfl_down(first, 1);  // the first start strictly after this token
  if (lane == 63) f = N;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    l = max(l, max(w_before[w], w < wave ? w_last[w] : -1));
    f = min(f, min(w_after[w], w > wave ? w_first[w] : N));
  }
  if (i < N) {
    lo[(int64_t)blockIdx.y * N + i] = l;
    hi[(int64_t)blockIdx.y * N + i] = f;
  }
}

// Padding mask (nonzero = real token): the row's real tokens [start, end) are one segment, every
// other token is padding (lo = hi = its index). bad[row] = 1 where the real tokens are not one run.
__global__ __launch_bounds__(kTpb) void seg_mask_kernel(const uint8_t* mask, int64_t row_stride, int N, int* lo, int* hi,
                                                        int* bad) {
  __shared__ int w_start[kWaves], w_end[kWaves], w_count[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint8_t* row = mask + (int64_t)blockIdx.y * row_stride;
  int start = N, end = 0, count = 0;
  scan_row(N, tid, [&](int i) {
    const bool real = row[i] != 0;
    start = min(start, real ? i : N);
    end = max(end, real ? i + 1 : 0);
    count += real;
  });
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    start = min(start, __shfl_xor(start, m));
    end = max(end, __shfl_xor(end, m));
    count += __shfl_xor(count, m);
  }
  if (lane == 0) {
    w_start[wave] = start;
    w_end[wave] = end;
    w_count[wave] = count;
  }
  __syncthreads();
  start = N;
  end = 0;
  count = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    start = min(start, w_start[w]);
    end = max(end, w_end[w]);
    count += w_count[w];
  }
  const int i = blockIdx.x * kTpb + tid;
  if (i < N) {
    const bool real = row[i] != 0;
    lo[(int64_t)blockIdx.y * N + i] = real ? start : i;
    hi[(int64_t)blockIdx.y * N + i] = real ? end : i;
  }
  if (blockIdx.x == 0 && tid == 0) bad[blockIdx.y] = count > 0 && count != end - start;
}

template __global__ void seg_positions_kernel<int64_t>(const int64_t*, int64_t, int, int*, int*);
template __global__ void seg_positions_kernel<int32_t>(const int32_t*, int64_t, int, int*, int*);

hipError_t launch_seg_positions(const void* pos, bool is64, int64_t row_stride, int B, int N, int* lo, int* hi,
                                hipStream_t stream) {
  const dim3 grid((N + kTpb - 1) / kTpb, B);
  if (is64) {
    hipLaunchKernelGGL(seg_positions_kernel<int64_t>, grid, dim3(kTpb), 0, stream, static_cast<const int64_t*>(pos),
                       row_stride, N, lo, hi);
  } else {
    hipLaunchKernelGGL(seg_positions_kernel<int32_t>, grid, dim3(kTpb), 0, stream, static_cast<const int32_t*>(pos),
                       row_stride, N, lo, hi);
  }
  return hipGetLastError();
}

hipError_t launch_seg_mask(const uint8_t* mask, int64_t row_stride, int B, int N, int* lo, int* hi, int* bad,
                           hipStream_t stream) {
  hipLaunchKernelGGL(seg_mask_kernel, dim3((N + kTpb - 1) / kTpb, B), dim3(kTpb), 0, stream, mask, row_stride, N, lo, hi,
                     bad);
  return hipGetLastError();
}

}  // namespace gfa
