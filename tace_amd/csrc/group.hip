// Stable grouping of integer keys (the receiver and sender CSRs of an edge
// list): positions 0 .. n-1 ordered by key, in position order within a key,
// and each key's range.  A counting sort: count (each position's place among
// its key's, in arrival order), scan, scatter, then every position is moved
// to its rank by id inside its key's range.  The degrees of a neighbour list
// are tens to hundreds, so the ranking reads each range a few dozen times
// from L1 and L2, where a radix or merge sort and a binary search take 10 to
// 30 launches.  Measured against those (us): the sender CSR of 46k edges of
// 1,024 nodes 58 -> 25, of 1.06 M edges of 12,288 nodes 124 -> 71; the
// receiver and sender CSR of shuffled edges 291 -> 81 and 607 -> 221 (with
// the checks; one wait for the host instead of three); 5.6 M edges of 101k
// nodes 261 (random keys of that size, which no neighbour list has, 282 ->
// 552: the counting atomics then miss L2).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tace_hip.h"
#include "scan.h"

int tace_fail_msg(const char* msg);   // tace_hip.hip
int tace_check_launch(const char* what);

namespace {

// ranges longer than this are ordered by a workgroup that walks all keys
// (k_group_long) instead of a rank per entry, whose cost grows with the
// square of the range
constexpr int LONG_RANGE = 4096;

// the keys, and (other != null) a second array of the same range that is only
// checked and converted (an edge list's senders beside its receivers)
template <typename K>
struct Keys {
  const K* keys;
  int64_t stride;
  const int* through;
  const K* other;
  int64_t ostride;
  int* other32;

  // key i as an int, -1 outside [0, n_keys); flags[0]: some key (or other
  // key) outside, flags[1]: keys not ascending
  __device__ __forceinline__ int get(int i, int n_keys, int* flags) const {
    const int64_t p = through ? through[i] : i;
    const K k = keys[p * stride];
    bool ok = k >= 0 && k < (K)n_keys;
    if (!ok) flags[0] = 1;
    if (i > 0 && keys[(through ? (int64_t)through[i - 1] : p - 1) * stride] > k) flags[1] = 1;
    if (other) {
      const K o = other[i * ostride];
      other32[i] = (int)o;
      if (o < 0 || o >= (K)n_keys) flags[0] = 1;
    }
    return ok ? (int)k : -1;
  }
};

template <typename K>
__global__ __launch_bounds__(256) void k_group_count(Keys<K> in, int n, int n_keys, int* __restrict__ k32,
                                                     int* __restrict__ cnt, int* __restrict__ place,
                                                     int* __restrict__ flags) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  const int key = in.get(i, n_keys, flags);
  k32[i] = key;
  if (key >= 0) place[i] = atomicAdd(cnt + key, 1);
}

__global__ __launch_bounds__(1024) void k_group_scan(const int* __restrict__ cnt, int m, int* __restrict__ out) {
  scan_1024(cnt, m, out);
}

__global__ __launch_bounds__(256) void k_group_scatter(const int* __restrict__ k32, const int* __restrict__ place,
                                                       int n, const int* __restrict__ rowptr, int* __restrict__ tmp) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i >= n || k32[i] < 0) return;
  tmp[rowptr[k32[i]] + place[i]] = i;
}

__global__ __launch_bounds__(256) void k_group_rank(const int* __restrict__ k32, int n, const int* __restrict__ rowptr,
                                                    const int* __restrict__ tmp, int* __restrict__ order) {
  const int q = (int)(blockIdx.x * 256 + threadIdx.x);
  if (q >= n) return;
  const int i = tmp[q];
  if (i < 0) return;   // a position whose key was out of range left its slot empty
  const int key = k32[i], b = rowptr[key], e = rowptr[key + 1];
  if (e - b > LONG_RANGE) return;
  int r = b;
#pragma unroll 4
  for (int p = b; p < e; ++p) r += tmp[p] < i;
  order[r] = i;
}

// the ranges longer than LONG_RANGE: each holds a multiple of LONG_RANGE; the
// workgroup of the first one walks all keys and keeps the range's in order
__global__ __launch_bounds__(1024) void k_group_long(const int* __restrict__ k32, int n, const int* __restrict__ rowptr,
                                                     const int* __restrict__ tmp, int* __restrict__ order) {
  __shared__ int wcnt[16];
  const int q = (int)blockIdx.x * LONG_RANGE;
  if (q >= n) return;
  const int i0 = tmp[q];
  if (i0 < 0) return;
  const int key = k32[i0], b = rowptr[key], e = rowptr[key + 1];
  if (e - b <= LONG_RANGE || q - LONG_RANGE >= b) return;   // short, or another workgroup's
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
  int at = b;
  for (int p = 0; p < n; p += 1024) {
    const bool hit = p + t < n && k32[p + t] == key;
    const unsigned long long mask = __ballot(hit);
    if (lane == 0) wcnt[w] = __popcll(mask);
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k < w) before += wcnt[k];
      total += wcnt[k];
    }
    if (hit) order[at + before + __popcll(mask & ((1ull << lane) - 1))] = p + t;
    at += total;
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void k_group_fill(int* __restrict__ a, int64_t na, int va, int* __restrict__ b,
                                                    int64_t nb, int vb) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < na) a[i] = va;
  if (i < nb) b[i] = vb;
}

// All of it in one workgroup for few positions (counts, places and ranges in
// LDS): below SMALL_N the launches, not the work, take the time.
constexpr int SMALL_N = 8192, SMALL_KEYS = 4096;

template <typename K>
__global__ __launch_bounds__(1024) void k_group_small(Keys<K> in, int n, int n_keys, int* __restrict__ k32,
                                                      int* __restrict__ rowptr, int* __restrict__ order,
                                                      int* __restrict__ flags) {
  __shared__ int cnt[SMALL_KEYS], start[SMALL_KEYS + 1], tmp[SMALL_N], wsum[16], fl[2];
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
  for (int i = t; i < n_keys; i += 1024) cnt[i] = 0;
  if (t < 2) fl[t] = 0;
  __syncthreads();
  constexpr int PER = SMALL_N / 1024;
  int key[PER], place[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = t + 1024 * u;
    key[u] = -1;
    if (i < n) {
      k32[i] = key[u] = in.get(i, n_keys, fl);
      if (key[u] >= 0) place[u] = atomicAdd(&cnt[key[u]], 1);
    }
  }
  __syncthreads();
  // exclusive scan of cnt: four counts per thread
  {
    int v[4], s = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = 4 * t + q < n_keys ? cnt[4 * t + q] : 0;
      s += v[q];
    }
    int inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(inc, o, 64);
      if (lane >= o) inc += x;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int run = inc - s, total = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k < w) run += wsum[k];
      total += wsum[k];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (4 * t + q < n_keys) start[4 * t + q] = rowptr[4 * t + q] = run;
      run += v[q];
    }
    if (t == 0) start[n_keys] = rowptr[n_keys] = total;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u)
    if (key[u] >= 0) tmp[start[key[u]] + place[u]] = t + 1024 * u;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    if (key[u] < 0) continue;
    const int i = t + 1024 * u, e = start[key[u] + 1];
    int r = start[key[u]];
    for (int p = start[key[u]]; p < e; ++p) r += tmp[p] < i;
    order[r] = i;
  }
  if (t < 2 && flags) flags[t] = fl[t];
}

template <typename K>
int group_keys(const Keys<K>& in, int n, int n_keys, int32_t* k32, int32_t* rowptr, int32_t* order, int32_t* work,
               int32_t* flags, hipStream_t s) {
  if (n <= SMALL_N && n_keys <= SMALL_KEYS) {
    hipLaunchKernelGGL(k_group_small<K>, dim3(1), dim3(1024), 0, s, in, n, n_keys, k32, rowptr, order, flags);
    return tace_check_launch("tace_group_keys");
  }
  int* cnt = work;            // n_keys, then two flags when the caller wants none
  int* fl = cnt + n_keys;
  int* place = fl + 2;        // n
  int* tmp = place + n;       // n
  int* f = flags ? flags : fl;
  const unsigned nb = (unsigned)((n + 255) / 256);
  const int64_t most = n_keys + 2 > n ? (int64_t)n_keys + 2 : n;
  hipLaunchKernelGGL(k_group_fill, dim3((unsigned)((most + 255) / 256)), dim3(256), 0, s, cnt, (int64_t)n_keys + 2, 0,
                     tmp, (int64_t)n, -1);
  if (flags) hipLaunchKernelGGL(k_group_fill, dim3(1), dim3(256), 0, s, flags, (int64_t)2, 0, flags, (int64_t)0, 0);
  if (n > 0)
    hipLaunchKernelGGL(k_group_count<K>, dim3(nb), dim3(256), 0, s, in, n, n_keys, k32, cnt, place, f);
  hipLaunchKernelGGL(k_group_scan, dim3(1), dim3(1024), 0, s, cnt, n_keys, rowptr);
  if (n > 0) {
    hipLaunchKernelGGL(k_group_scatter, dim3(nb), dim3(256), 0, s, k32, place, n, rowptr, tmp);
    hipLaunchKernelGGL(k_group_rank, dim3(nb), dim3(256), 0, s, k32, n, rowptr, tmp, order);
    if (n > LONG_RANGE)
      hipLaunchKernelGGL(k_group_long, dim3((unsigned)((n + LONG_RANGE - 1) / LONG_RANGE)), dim3(1024), 0, s, k32, n,
                         rowptr, tmp, order);
  }
  return tace_check_launch("tace_group_keys");
}

}  // namespace

extern "C" int64_t tace_group_keys_work(int64_t n, int64_t n_keys) { return 2 * n + n_keys + 4; }

extern "C" int tace_group_keys(int key_bytes, const void* keys, int64_t stride, const int32_t* through, int64_t n,
                               int64_t n_keys, int32_t* keys32, int32_t* rowptr, int32_t* order, const void* other,
                               int64_t other_stride, int32_t* other32, int32_t* work, int32_t* flags, void* stream) {
  if (n < 0 || n_keys < 0 || n > INT32_MAX - 8192 || n_keys > INT32_MAX - 8192)
    return tace_fail_msg("tace_group_keys: bad sizes");
  if (!rowptr || !work || (n && (!keys || !keys32 || !order)) || (other && !other32))
    return tace_fail_msg("tace_group_keys: null pointer");
  hipStream_t s = (hipStream_t)stream;
  if (key_bytes == 8) {
    const Keys<int64_t> in{(const int64_t*)keys, stride, through, (const int64_t*)other, other_stride, other32};
    return group_keys(in, (int)n, (int)n_keys, keys32, rowptr, order, work, flags, s);
  }
  if (key_bytes == 4) {
    const Keys<int32_t> in{(const int32_t*)keys, stride, through, (const int32_t*)other, other_stride, other32};
    return group_keys(in, (int)n, (int)n_keys, keys32, rowptr, order, work, flags, s);
  }
  return tace_fail_msg("tace_group_keys: keys of 4 or 8 bytes");
}
