// Stable grouping of integer keys (the receiver and sender CSRs of an edge
// list): positions 0 .. n-1 ordered by key, in position order within a key,
// and each key's range.  A radix sort from the low digit that moves (key,
// position) pairs only: per digit a workgroup counts its 2,048 positions in
// LDS, one scan per digit value turns the counts into places, and a position's
// rank among the equal digits of its wavefront comes from ballots.  No atomic
// reaches memory and no step depends on how the keys are distributed.  (A
// counting sort by atomics, ranking every range by its length squared, was
// faster at best and did not have that: atomics on neighbouring keys meet in
// one slice of the memory, a hub or a handful of keys makes the ranges long.)
//
// us, library sort and binary search | that counting sort | this: senders of
// fcc lists of 78 edges a node, 13,500 nodes 124 | 81 | 51, with node ids
// shuffled 124 | 163 | 58; 97,556 nodes shuffled 362 | 751 | 289; 8,192 equal
// keys 41 | 3,129 | 15; 361,000 sorted under 16 keys 120 | 4,296 | 22; 30 M
// random under 1 M keys 1,431 | 3,473 | 1,002.  The receiver CSR of 1.05 M
// edges with the checks and the host's wait, sorted 228 | 253 | 78, shuffled
// 459 | 133 | 87 (bincount, two minima, argsort before).  A few microseconds
// per launch at 300,000 edges, latency; what the loads of a thread wait for
// together decides the large sizes (97,556 nodes shuffled: 395 one by one).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tace_hip.h"
#include "scan.h"

int tace_fail_msg(const char* msg);   // tace_hip.hip
int tace_check_launch(const char* what);

namespace {

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

  struct Loaded {
    K key, before, other;   // key i, key i - 1, other key i
  };

  __device__ __forceinline__ Loaded load(int i) const {
    const int64_t p = through ? through[i] : i, q = i == 0 ? p : through ? (int64_t)through[i - 1] : p - 1;
    return {keys[p * stride], keys[q * stride], other ? other[i * ostride] : (K)0};
  }

  // key i as an int, -1 outside [0, n_keys); flags[0]: some key (or other
  // key) outside, flags[1]: keys not ascending
  __device__ __forceinline__ int take(const Loaded& v, int i, int n_keys, int* flags) const {
    bool ok = v.key >= 0 && v.key < (K)n_keys;
    if (v.before > v.key) flags[1] = 1;
    if (other) other32[i] = (int)v.other;
    if (!ok || (other && (v.other < 0 || v.other >= (K)n_keys))) flags[0] = 1;
    return ok ? (int)v.key : -1;
  }
};

// keys outside the range come after all others
__device__ __forceinline__ int sort_key(int k32, int n_keys) { return k32 < 0 ? n_keys : k32; }

// the lanes that hold this lane's digit (of `bits` bits), of those with in
__device__ __forceinline__ unsigned long long same_digit(int d, int bits, bool in) {
  unsigned long long m = __ballot(in);
  for (int b = 0; b < bits; ++b) {
    const bool one = (d >> b) & 1;
    const unsigned long long v = __ballot(one);
    m &= one ? v : ~v;
  }
  return m;
}

// this lane's place among its wavefront's equal digits so far: cnt[d] holds
// them and grows by this step's
__device__ __forceinline__ int digit_rank(int* cnt, int d, int bits, bool in, int lane) {
  const unsigned long long m = same_digit(d, bits, in);
  const int r = __popcll(m & ((1ull << lane) - 1));
  int before = 0;
  if (in && r == 0) before = atomicAdd(cnt + d, __popcll(m));
  return r + __shfl(before, in ? __ffsll((long long)m) - 1 : lane, 64);
}

constexpr int MAX_BITS = 9, MAX_BINS = 1 << MAX_BITS;   // a digit's
// positions a workgroup: a run of 64 STEPS per wavefront, whose ranks are a
// serial chain (1.05 M edges, 2 digits, loads one by one: 57 us; 16 steps 71,
// 32 steps 101)
constexpr int STEPS = 8, CHUNK = 256 * STEPS;

// Counts of the lowest digit per workgroup, hist [bins + 2][nwg]; the last two
// rows hold the flags.  Reads, checks and converts the keys.
template <typename K>
__global__ __launch_bounds__(256) void k_group_first(Keys<K> in, int n, int n_keys, int bins, int* __restrict__ k32,
                                                     int* __restrict__ hist) {
  __shared__ int cnt[MAX_BINS + 2];
  const int t = (int)threadIdx.x;
  for (int b = t; b < bins + 2; b += 256) cnt[b] = 0;
  __syncthreads();
  // every load goes out before the first is waited for (past the end: the last key)
  const int64_t i0 = (int64_t)blockIdx.x * CHUNK + t;
  typename Keys<K>::Loaded v[STEPS];
#pragma unroll
  for (int u = 0; u < STEPS; ++u) v[u] = in.load((int)min(i0 + 256 * u, (int64_t)n - 1));
#pragma unroll
  for (int u = 0; u < STEPS; ++u) {
    if (i0 + 256 * u >= n) break;
    const int i = (int)i0 + 256 * u, key = in.take(v[u], i, n_keys, cnt + bins);
    k32[i] = key;
    atomicAdd(cnt + (sort_key(key, n_keys) & (bins - 1)), 1);
  }
  __syncthreads();
  for (int b = t; b < bins + 2; b += 256) hist[(int64_t)b * gridDim.x + blockIdx.x] = cnt[b];
}

// the same of a later digit (no flags)
__global__ __launch_bounds__(256) void k_group_count(const int* __restrict__ keys, int n, int shift, int bins,
                                                     int* __restrict__ hist) {
  __shared__ int cnt[MAX_BINS];
  const int t = (int)threadIdx.x;
  for (int b = t; b < bins; b += 256) cnt[b] = 0;
  __syncthreads();
  const int64_t i0 = (int64_t)blockIdx.x * CHUNK + t;
  int v[STEPS];
#pragma unroll
  for (int u = 0; u < STEPS; ++u) v[u] = keys[min(i0 + 256 * u, (int64_t)n - 1)];
#pragma unroll
  for (int u = 0; u < STEPS; ++u)
    if (i0 + 256 * u < n) atomicAdd(cnt + ((v[u] >> shift) & (bins - 1)), 1);
  __syncthreads();
  for (int b = t; b < bins; b += 256) hist[(int64_t)b * gridDim.x + blockIdx.x] = cnt[b];
}

// a workgroup per digit value: its counts before each workgroup, offs [bins +
// 2][nwg + 1], the last column their total; flags from the two rows after them
__global__ __launch_bounds__(1024) void k_group_scan(const int* __restrict__ hist, int nwg, int bins,
                                                     int* __restrict__ offs, int* __restrict__ flags) {
  int* o = offs + (int64_t)blockIdx.x * (nwg + 1);
  scan_1024(hist + (int64_t)blockIdx.x * nwg, nwg, o);
  if (flags && (int)blockIdx.x >= bins && threadIdx.x == 0) flags[blockIdx.x - bins] = o[nwg] != 0;
}

// Every (key, position) to its place by one digit.  pos null: position i is i.
__global__ __launch_bounds__(256) void k_group_scatter(const int* __restrict__ keys, const int* __restrict__ pos, int n,
                                                       int n_keys, int shift, int bits, const int* __restrict__ offs,
                                                       int* __restrict__ keys_out, int* __restrict__ pos_out) {
  __shared__ int cnt[4][MAX_BINS], total[MAX_BINS], before[MAX_BINS], wsum[4];
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6, bins = 1 << bits, nwg = (int)gridDim.x;
  for (int b = t; b < bins; b += 256) cnt[0][b] = cnt[1][b] = cnt[2][b] = cnt[3][b] = 0;
  const int64_t i0 = (int64_t)blockIdx.x * CHUNK + 64 * STEPS * w + lane;
  int key[STEPS], rank[STEPS], at0[STEPS];
#pragma unroll
  for (int u = 0; u < STEPS; ++u) {
    const int64_t i = min(i0 + 64 * u, (int64_t)n - 1);
    key[u] = keys[i];
    at0[u] = pos ? pos[i] : (int)i;
  }
  for (int b = t; b < bins; b += 256) {
    total[b] = offs[(int64_t)b * (nwg + 1) + nwg];
    before[b] = offs[(int64_t)b * (nwg + 1) + blockIdx.x];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < STEPS; ++u) {
    key[u] = i0 + 64 * u < n ? sort_key(key[u], n_keys) : -1;
    rank[u] = digit_rank(cnt[w], (key[u] >> shift) & (bins - 1), bits, key[u] >= 0, lane);
  }
  // where each digit's positions of each wavefront go: all smaller digits,
  // the digit's in the workgroups before, in the wavefronts before.  Thread t
  // has digits 2 t and 2 t + 1.
  const int s = (2 * t < bins ? total[2 * t] : 0) + (2 * t + 1 < bins ? total[2 * t + 1] : 0);
  int inc = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(inc, o, 64);
    if (lane >= o) inc += x;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int run = inc - s;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k < w) run += wsum[k];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int b = 2 * t + q;
    if (b < bins) {
      int at = run + before[b];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int c = cnt[k][b];
        cnt[k][b] = at;
        at += c;
      }
      run += total[b];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < STEPS; ++u) {
    if (key[u] < 0) continue;
    const int at = cnt[w][(key[u] >> shift) & (bins - 1)] + rank[u];
    keys_out[at] = key[u];
    pos_out[at] = at0[u];
  }
}

// rowptr[k] = the number of sorted keys below k
__global__ __launch_bounds__(256) void k_group_rows(const int* __restrict__ sorted, int n, int n_keys,
                                                    int* __restrict__ rowptr) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k > n_keys) return;
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = lo + (hi - lo) / 2;
    if (sorted[mid] < k) lo = mid + 1;
    else hi = mid;
  }
  rowptr[k] = lo;
}

// All of it in one workgroup for few positions, (key, position) packed in one
// word and kept in LDS: below SMALL_N the launches, not the work, take the time.
constexpr int SMALL_N = 8192, SMALL_KEYS = 4096, POS_BITS = 13, SMALL_BITS = 7, SMALL_BINS = 1 << SMALL_BITS;

template <typename K>
__global__ __launch_bounds__(1024) void k_group_small(Keys<K> in, int n, int n_keys, int bits, int passes,
                                                      int* __restrict__ k32, int* __restrict__ rowptr,
                                                      int* __restrict__ order, int* __restrict__ flags) {
  __shared__ int data[SMALL_N], cnt[16][SMALL_BINS], wsum[16], fl[2];
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6, bins = 1 << bits;
  // each wavefront a run of 64 `steps` positions: all of them take part however
  // few there are, as the steps are serial (1,792 edges: 12 us with 8 steps)
  constexpr int PER = SMALL_N / 1024;
  const int steps = (n + 1023) >> 10;
  if (t < 2) fl[t] = 0;
  __syncthreads();
  const int i0 = 64 * steps * w + lane;
  int v[PER], rank[PER];
  {
    typename Keys<K>::Loaded l[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u)
      if (u < steps) l[u] = in.load(min(i0 + 64 * u, n - 1));   // (no steps without positions)
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = i0 + 64 * u;
      v[u] = -1;
      if (u < steps && i < n) {
        const int key = in.take(l[u], i, n_keys, fl);
        k32[i] = key;
        v[u] = (sort_key(key, n_keys) << POS_BITS) | i;
      }
    }
  }
  for (int p = 0; p < passes; ++p) {
    const int shift = POS_BITS + p * bits;
    for (int b = t; b < 16 * SMALL_BINS; b += 1024) cnt[b / SMALL_BINS][b % SMALL_BINS] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u)
      if (u < steps) rank[u] = digit_rank(cnt[w], (v[u] >> shift) & (bins - 1), bits, v[u] >= 0, lane);
    __syncthreads();
    // exclusive scan over (digit, wavefront): thread t has two wavefronts'
    // counts of digit t / 8
    int* c = &cnt[2 * (t & 7)][t >> 3];
    const int a0 = c[0], a1 = c[SMALL_BINS], s = a0 + a1;
    int inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(inc, o, 64);
      if (lane >= o) inc += x;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int run = inc - s;
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (k < w) run += wsum[k];
    c[0] = run;
    c[SMALL_BINS] = run + a0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u)
      if (v[u] >= 0) data[cnt[w][(v[u] >> shift) & (bins - 1)] + rank[u]] = v[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u) v[u] = u < steps && i0 + 64 * u < n ? data[i0 + 64 * u] : -1;
    // (the next pass's barriers keep its writes of data behind these reads)
  }
#pragma unroll
  for (int u = 0; u < PER; ++u)
    if (v[u] >= 0) order[i0 + 64 * u] = v[u] & (SMALL_N - 1);
  for (int k = t; k <= n_keys; k += 1024) {
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if ((data[mid] >> POS_BITS) < k) lo = mid + 1;
      else hi = mid;
    }
    rowptr[k] = lo;
  }
  if (t < 2 && flags) flags[t] = fl[t];
}

// digits of at most `most` bits for sort keys 0 .. n_keys
void digits(int n_keys, int most, int* bits, int* passes) {
  int nb = 1;
  while (nb < 31 && (n_keys >> nb) != 0) ++nb;
  *passes = (nb + most - 1) / most;
  *bits = (nb + *passes - 1) / *passes;
}

template <typename K>
int group_keys(const Keys<K>& in, int n, int n_keys, int32_t* k32, int32_t* rowptr, int32_t* order, int32_t* work,
               int32_t* flags, hipStream_t s) {
  int bits, passes;
  if (n <= SMALL_N && n_keys <= SMALL_KEYS) {
    digits(n_keys, SMALL_BITS, &bits, &passes);
    hipLaunchKernelGGL(k_group_small<K>, dim3(1), dim3(1024), 0, s, in, n, n_keys, bits, passes, k32, rowptr, order,
                       flags);
    return tace_check_launch("tace_group_keys");
  }
  digits(n_keys, MAX_BITS, &bits, &passes);
  const int bins = 1 << bits, nwg = n / CHUNK + (n % CHUNK != 0);
  // the last pass writes (sorted, order), the ones before it alternate between
  // that and (keys_b, pos_b); none reads what it writes
  int* sorted = work;
  int* keys_b = sorted + n;
  int* pos_b = keys_b + n;
  int* hist = pos_b + n;                              // (bins + 2) nwg
  int* offs = hist + (int64_t)(bins + 2) * nwg;       // (bins + 2) (nwg + 1)
  const int *keys = k32, *pos = nullptr;
  if (n == 0 && flags) {   // (the flags of no keys)
    hipLaunchKernelGGL(k_group_scan, dim3(2), dim3(1024), 0, s, hist, 0, 0, offs, flags);
  }
  for (int p = 0; p < passes && n > 0; ++p) {
    const bool last = ((passes - 1 - p) & 1) == 0;
    int *ko = last ? sorted : keys_b, *po = last ? order : pos_b;
    if (p == 0)
      hipLaunchKernelGGL(k_group_first<K>, dim3((unsigned)nwg), dim3(256), 0, s, in, n, n_keys, bins, k32, hist);
    else
      hipLaunchKernelGGL(k_group_count, dim3((unsigned)nwg), dim3(256), 0, s, keys, n, p * bits, bins, hist);
    hipLaunchKernelGGL(k_group_scan, dim3((unsigned)(p == 0 ? bins + 2 : bins)), dim3(1024), 0, s, hist, nwg, bins,
                       offs, flags);
    hipLaunchKernelGGL(k_group_scatter, dim3((unsigned)nwg), dim3(256), 0, s, keys, pos, n, n_keys, p * bits, bits,
                       offs, ko, po);
    keys = ko;
    pos = po;
  }
  hipLaunchKernelGGL(k_group_rows, dim3((unsigned)(n_keys / 256 + 1)), dim3(256), 0, s, sorted, n, n_keys, rowptr);
  return tace_check_launch("tace_group_keys");
}

}  // namespace

extern "C" int64_t tace_group_keys_work(int64_t n, int64_t n_keys) {
  // three arrays of n and the counts of MAX_BINS digit values and two flags
  // per workgroup before and after their scan
  (void)n_keys;
  const int64_t nwg = (n + CHUNK - 1) / CHUNK;
  return 3 * n + (MAX_BINS + 2) * (2 * nwg + 1);
}

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
