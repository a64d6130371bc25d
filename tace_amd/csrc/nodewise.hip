// Node-wise glue of the model in one pass over memory each: the gate
// nonlinearity and the energy readout, forward and input gradient.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tace_hip.h"
#include "common.h"

int tace_fail_msg(const char* msg);   // tace_hip.hip
int tace_check_launch(const char* what);

namespace {

template <typename T, int V>
struct Vec {
  typedef T type __attribute__((ext_vector_type(V)));
};
template <typename T>
struct Vec<T, 1> {
  typedef T type;
};

template <typename T>
__device__ __forceinline__ T sigmoid_of(T v) {
  return T(1) / (T(1) + exp(-v));
}

template <typename T, int V>
__device__ __forceinline__ typename Vec<T, V>::type sigmoid_vec(typename Vec<T, V>::type v) {
  if constexpr (V == 1) {
    return sigmoid_of(v);
  } else {
    typename Vec<T, V>::type r;
#pragma unroll
    for (int i = 0; i < V; ++i) r[i] = sigmoid_of(v[i]);
    return r;
  }
}

// The gate of NB blocks l = 0 .. NB - 1 of C channels on group-major features:
// x is [n, (NB + 1) C] (the gates, one C-run per block, then the l = 0
// features) followed by the blocks [n, 2l + 1, C] of l >= 1; out_l = cst
// sigmoid(gate_l) x_l, the blocks [n, 2l + 1, C] one after the other.
//
// A thread takes V adjacent channels of one node through all blocks, so every
// value is read and written once; what bounds it is that traffic.  As torch
// operations it was 6 launches forward and 16 backward, which read the gate
// activations and products back in between: 12,288 nodes, L = 3, C = 128
// (227 MB forward, 353 MB backward): forward 74 -> 33 us, backward 178 -> 74
// us; at 1,024 nodes the launches themselves were the cost (69 -> 14 us and
// 179 -> 69 us with the host's share).
template <typename T, int V, int NB>
__global__ __launch_bounds__(256) void k_gate_fwd(const T* __restrict__ x, int64_t n, int C, T cst,
                                                  T* __restrict__ out) {
  typedef typename Vec<T, V>::type vec;
  const int per = C / V;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t a = id / per;
  if (a >= n) return;
  const int c = (int)(id - a * per) * V;
  const T* x0 = x + a * (NB + 1) * C + c;
  vec g[NB];
#pragma unroll
  for (int l = 0; l < NB; ++l) g[l] = *(const vec*)(x0 + l * C);
  vec f[NB * NB];
  f[0] = *(const vec*)(x0 + NB * C);
  const T* xb = x + n * (NB + 1) * C;   // block l >= 1 starts at n C (l^2 - 1) past this
#pragma unroll
  for (int l = 1; l < NB; ++l)
#pragma unroll
    for (int m = 0; m < 2 * l + 1; ++m)
      f[l * l + m] = *(const vec*)(xb + n * C * (l * l - 1) + (a * (2 * l + 1) + m) * C + c);
#pragma unroll
  for (int l = 0; l < NB; ++l) {
    const vec s = cst * sigmoid_vec<T, V>(g[l]);
#pragma unroll
    for (int m = 0; m < 2 * l + 1; ++m) *(vec*)(out + n * C * l * l + (a * (2 * l + 1) + m) * C + c) = s * f[l * l + m];
  }
}

// its input gradient: g_x_l = g_out_l cst sigmoid(gate_l); the gate's is cst
// sigmoid' times the sum over the block's components of g_out x
template <typename T, int V, int NB>
__global__ __launch_bounds__(256) void k_gate_bwd(const T* __restrict__ x, const T* __restrict__ go, int64_t n, int C,
                                                  T cst, T* __restrict__ gx) {
  typedef typename Vec<T, V>::type vec;
  const int per = C / V;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t a = id / per;
  if (a >= n) return;
  const int c = (int)(id - a * per) * V;
  const T* x0 = x + a * (NB + 1) * C + c;
  T* g0 = gx + a * (NB + 1) * C + c;
  const T* xb = x + n * (NB + 1) * C;
  T* gb = gx + n * (NB + 1) * C;
#pragma unroll
  for (int l = 0; l < NB; ++l) {
    const vec s = sigmoid_vec<T, V>(*(const vec*)(x0 + l * C));
    vec dot = vec(T(0));
#pragma unroll
    for (int m = 0; m < 2 * l + 1; ++m) {
      const int64_t o = (a * (2 * l + 1) + m) * C + c, ob = n * C * (l * l - 1) + o;
      const vec g = *(const vec*)(go + n * C * l * l + o);
      const vec v = l == 0 ? *(const vec*)(x0 + NB * C) : *(const vec*)(xb + ob);
      dot += g * v;
      *(vec*)(l == 0 ? g0 + NB * C : gb + ob) = cst * s * g;
    }
    *(vec*)(g0 + l * C) = cst * s * (T(1) - s) * dot;
  }
}

template <typename T, int V, bool BWD>
int gate_launch(int nb, const T* x, const T* go, int64_t n, int C, T cst, T* out, hipStream_t s) {
  const int64_t threads = n * (C / V);
  const dim3 g((unsigned)((threads + 255) / 256)), b(256);
#define GATE_CASE(NB)                                                                    \
  case NB:                                                                               \
    if constexpr (BWD) hipLaunchKernelGGL((k_gate_bwd<T, V, NB>), g, b, 0, s, x, go, n, C, cst, out); \
    else hipLaunchKernelGGL((k_gate_fwd<T, V, NB>), g, b, 0, s, x, n, C, cst, out);        \
    break;
  switch (nb) {
    GATE_CASE(1)
    GATE_CASE(2)
    GATE_CASE(3)
    GATE_CASE(4)
    default: return tace_fail_msg("tace_gate: 1..4 blocks");
  }
#undef GATE_CASE
  return tace_check_launch("tace_gate");
}

template <typename T, bool BWD>
int gate_any(int nb, const void* x, const void* go, int64_t n, int C, double cst, void* out, hipStream_t s) {
  constexpr int V = 16 / sizeof(T);
  // 16-byte accesses: every row and block starts on a multiple of C values
  if (C % V == 0 && ((((uintptr_t)x) | ((uintptr_t)go) | ((uintptr_t)out)) & 15) == 0)
    return gate_launch<T, V, BWD>(nb, (const T*)x, (const T*)go, n, C, (T)cst, (T*)out, s);
  return gate_launch<T, 1, BWD>(nb, (const T*)x, (const T*)go, n, C, (T)cst, (T*)out, s);
}

// The energy readout of a node: e = sum_j w2_j silu(sum_c x_c w1_cj), 16
// hidden values (w1 [C, 16] and w2 [16] carry their scales, the activation's
// constant is in w2).  One wavefront per node; lane l holds w1's rows l + 64 i
// for the nodes it goes through, the 16 sums come from a transposing
// butterfly.  For the input gradient hid[n, 16] keeps w2_j silu'(h_j).  Then
// the node's energy: vals[n] = (e0 . attrs, e scale . attrs + shift . attrs),
// scale and shift zero for an atom alone in its graph without edges.
//
// Bound by latency at every size of use (6 MB of x at 12,288 nodes): its
// worth is in the ~30 launches of torch operations and two GEMM launches it
// replaces: with the gate above, the grouping and the edge list's kernels an
// MD step of 1,024 atoms went from 214 to 121 launches and 3.86 to 2.85 ms.
constexpr int HEAD_H = 16, HEAD_MAXC = 512;

template <typename T, int NC>
__global__ __launch_bounds__(256) void k_energy_head(const T* __restrict__ x, const int64_t* __restrict__ row_of,
                                                     const T* __restrict__ w1, const T* __restrict__ w2, int64_t n,
                                                     int C, const T* __restrict__ attrs, int S,
                                                     const T* __restrict__ e0, const T* __restrict__ scale,
                                                     const T* __restrict__ shift, const int64_t* __restrict__ batch,
                                                     const int64_t* __restrict__ ptr, const int* __restrict__ rowptr,
                                                     T* __restrict__ hid, T* __restrict__ vals,
                                                     T* __restrict__ fac, T* __restrict__ enode) {
  const int lane = (int)threadIdx.x & 63;
  const int64_t w0 = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), nw = (int64_t)gridDim.x * 4;
  T wr[NC][HEAD_H];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = lane + 64 * i;
#pragma unroll
    for (int j = 0; j < HEAD_H; ++j) wr[i][j] = c < C ? w1[(int64_t)c * HEAD_H + j] : T(0);
  }
  const int jl = rev4(lane);   // the hidden value this lane holds after the butterfly
  const T w2j = w2[jl];
  for (int64_t a = w0; a < n; a += nw) {
    const int64_t r = row_of[a];
    T h[HEAD_H];
#pragma unroll
    for (int j = 0; j < HEAD_H; ++j) h[j] = T(0);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      const T v = c < C ? x[r * C + c] : T(0);
#pragma unroll
      for (int j = 0; j < HEAD_H; ++j) h[j] += v * wr[i][j];
    }
    const T hj = reduce16_lanes<T>(h[0], h[1], h[2], h[3], h[4], h[5], h[6], h[7], h[8], h[9], h[10], h[11], h[12],
                                   h[13], h[14], h[15]);
    const T s = sigmoid_of(hj);
    T e = w2j * hj * s;
    e += __shfl_xor(e, 1, 64);
    e += __shfl_xor(e, 2, 64);
    e += __shfl_xor(e, 4, 64);
    e += __shfl_xor(e, 8, 64);
    if (lane < HEAD_H) hid[a * HEAD_H + jl] = w2j * (s + hj * s * (T(1) - s));
    // the element tables' products with the node's attributes
    T b0 = T(0), sc = T(0), sh = T(0);
    for (int k = lane; k < S; k += 64) {
      const T v = attrs[a * S + k];
      b0 += v * e0[k];
      sc += v * scale[k];
      sh += v * shift[k];
    }
    b0 = wave_sum(b0);
    sc = wave_sum(sc);
    sh = wave_sum(sh);
    if (lane == 0) {
      const int64_t g = batch[a];
      if (ptr[g + 1] - ptr[g] == 1 && rowptr[a + 1] == rowptr[a]) sc = sh = T(0);
      const T m = e * sc + sh;
      vals[2 * a] = b0;
      vals[2 * a + 1] = m;
      fac[a] = sc;
      enode[a] = b0 + m;
    }
  }
}

// E[g] = sum of vals[., 0] + sum of vals[., 1] over the graph's nodes, each
// column in a fixed order (thread t takes nodes t + 1024 i, then a tree)
template <typename T>
__global__ __launch_bounds__(1024) void k_energy_sum(const T* __restrict__ vals, const int64_t* __restrict__ ptr,
                                                     T* __restrict__ E) {
  __shared__ T sh[2][16];
  const int t = (int)threadIdx.x;
  T a = T(0), b = T(0);
  for (int64_t k = ptr[blockIdx.x] + t; k < ptr[blockIdx.x + 1]; k += 1024) {
    a += vals[2 * k];
    b += vals[2 * k + 1];
  }
  a = wave_sum(a);
  b = wave_sum(b);
  if ((t & 63) == 0) {
    sh[0][t >> 6] = a;
    sh[1][t >> 6] = b;
  }
  __syncthreads();
  if (t == 0) {
    a = b = T(0);
    for (int w = 0; w < 16; ++w) {
      a += sh[0][w];
      b += sh[1][w];
    }
    E[blockIdx.x] = a + b;
  }
}

// g_x[row_of[n], c] = (g_E[graph of n] + g_node[n]) fac[n] sum_j hid[n, j] w1[c, j]
template <typename T, int NC>
__global__ __launch_bounds__(256) void k_energy_head_bwd(const T* __restrict__ hid, const T* __restrict__ fac,
                                                         const T* __restrict__ gE, const T* __restrict__ gnode,
                                                         const int64_t* __restrict__ row_of,
                                                         const int64_t* __restrict__ batch,
                                                         const T* __restrict__ w1, int64_t n, int C,
                                                         T* __restrict__ gx) {
  const int lane = (int)threadIdx.x & 63;
  const int64_t w0 = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), nw = (int64_t)gridDim.x * 4;
  T wr[NC][HEAD_H];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = lane + 64 * i;
#pragma unroll
    for (int j = 0; j < HEAD_H; ++j) wr[i][j] = c < C ? w1[(int64_t)c * HEAD_H + j] : T(0);
  }
  for (int64_t a = w0; a < n; a += nw) {
    T f = gE ? gE[batch[a]] : T(0);
    if (gnode) f += gnode[a];
    f *= fac[a];
    const T* d = hid + a * HEAD_H;
    const int64_t r = row_of[a];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      T acc = T(0);
#pragma unroll
      for (int j = 0; j < HEAD_H; ++j) acc += d[j] * wr[i][j];
      const int c = lane + 64 * i;
      if (c < C) gx[r * C + c] = f * acc;
    }
  }
}

#define HEAD_NC(C, CALL)                          \
  switch (((C) + 63) / 64) {                      \
    case 1: CALL(1); break;                       \
    case 2: CALL(2); break;                       \
    case 3:                                       \
    case 4: CALL(4); break;                       \
    default: CALL(8); break;                      \
  }

template <typename T>
int head_fwd(const void* x, const int64_t* row_of, const void* w1, const void* w2, int64_t n, int C, const void* attrs,
             int S, const void* e0, const void* scale, const void* shift, const int64_t* batch, const int64_t* ptr,
             const int32_t* rowptr, int64_t n_graphs, void* hid, void* vals, void* fac, void* enode, void* E,
             hipStream_t s) {
  // four nodes' worth of work per wavefront before another workgroup pays
  const int64_t wg = (n + 15) / 16;
  const dim3 g((unsigned)(wg < 2048 ? wg : 2048)), b(256);
#define HEAD_CALL(NC)                                                                                                \
  hipLaunchKernelGGL((k_energy_head<T, NC>), g, b, 0, s, (const T*)x, row_of, (const T*)w1, (const T*)w2, n, C,      \
                     (const T*)attrs, S, (const T*)e0, (const T*)scale, (const T*)shift, batch, ptr, rowptr,         \
                     (T*)hid, (T*)vals, (T*)fac, (T*)enode)
  if (n > 0) {
    HEAD_NC(C, HEAD_CALL)
    if (int rc = tace_check_launch("tace_energy_head_fwd")) return rc;
  }
#undef HEAD_CALL
  hipLaunchKernelGGL(k_energy_sum<T>, dim3((unsigned)n_graphs), dim3(1024), 0, s, (const T*)vals, ptr, (T*)E);
  return tace_check_launch("tace_energy_head_fwd");
}

template <typename T>
int head_bwd(const void* hid, const void* fac, const void* gE, const void* gnode, const int64_t* row_of,
             const int64_t* batch, const void* w1, int64_t n, int C, void* gx, hipStream_t s) {
  const int64_t wg = (n + 15) / 16;
  const dim3 g((unsigned)(wg < 2048 ? wg : 2048)), b(256);
#define HEAD_CALL(NC)                                                                                              \
  hipLaunchKernelGGL((k_energy_head_bwd<T, NC>), g, b, 0, s, (const T*)hid, (const T*)fac, (const T*)gE,           \
                     (const T*)gnode, row_of, batch, (const T*)w1, n, C, (T*)gx)
  HEAD_NC(C, HEAD_CALL)
#undef HEAD_CALL
  return tace_check_launch("tace_energy_head_bwd");
}

bool gate_sizes_ok(int dtype, int64_t n, int32_t C, int32_t nb) {
  // threads of one launch: at most n C
  return (dtype == TACE_F32 || dtype == TACE_F64) && n >= 0 && C > 0 && nb >= 1 && nb <= 4 && n <= (int64_t)1 << 30 &&
         n * C < (int64_t)1 << 38;
}

}  // namespace

extern "C" int tace_gate_fwd(int dtype, const void* x, int64_t n_nodes, int32_t channels, int32_t n_blocks, double cst,
                             void* out, void* stream) {
  if (!gate_sizes_ok(dtype, n_nodes, channels, n_blocks)) return tace_fail_msg("tace_gate_fwd: bad dtype or sizes");
  if (n_nodes == 0) return 0;
  if (!x || !out) return tace_fail_msg("tace_gate_fwd: null pointer");
  return dtype == TACE_F32 ? gate_any<float, false>(n_blocks, x, x, n_nodes, channels, cst, out, (hipStream_t)stream)
                           : gate_any<double, false>(n_blocks, x, x, n_nodes, channels, cst, out, (hipStream_t)stream);
}

extern "C" int tace_gate_bwd(int dtype, const void* x, const void* g_out, int64_t n_nodes, int32_t channels,
                             int32_t n_blocks, double cst, void* g_x, void* stream) {
  if (!gate_sizes_ok(dtype, n_nodes, channels, n_blocks)) return tace_fail_msg("tace_gate_bwd: bad dtype or sizes");
  if (n_nodes == 0) return 0;
  if (!x || !g_out || !g_x) return tace_fail_msg("tace_gate_bwd: null pointer");
  return dtype == TACE_F32 ? gate_any<float, true>(n_blocks, x, g_out, n_nodes, channels, cst, g_x, (hipStream_t)stream)
                           : gate_any<double, true>(n_blocks, x, g_out, n_nodes, channels, cst, g_x,
                                                    (hipStream_t)stream);
}

extern "C" int tace_energy_head_fwd(int dtype, const void* x, const int64_t* row_of, const void* w1, const void* w2,
                                    int64_t n_nodes, int32_t channels, const void* attrs, int32_t n_species,
                                    const void* e0, const void* scale, const void* shift, const int64_t* batch,
                                    const int64_t* ptr, const int32_t* rowptr, int64_t n_graphs, void* hid, void* vals,
                                    void* factor, void* node_energy, void* energy, void* stream) {
  if (n_nodes < 0 || n_nodes > ((int64_t)1 << 31) || channels <= 0 || channels > HEAD_MAXC || n_species <= 0 ||
      n_graphs < 0 || n_graphs > INT32_MAX)
    return tace_fail_msg("tace_energy_head_fwd: bad sizes (1..512 channels)");
  if (n_graphs == 0) return 0;
  if (!ptr || !energy || (n_nodes && (!x || !row_of || !w1 || !w2 || !attrs || !e0 || !scale || !shift || !batch ||
                                      !rowptr || !hid || !vals || !factor || !node_energy)))
    return tace_fail_msg("tace_energy_head_fwd: null pointer");
  hipStream_t s = (hipStream_t)stream;
  if (dtype == TACE_F32)
    return head_fwd<float>(x, row_of, w1, w2, n_nodes, channels, attrs, n_species, e0, scale, shift, batch, ptr, rowptr,
                           n_graphs, hid, vals, factor, node_energy, energy, s);
  if (dtype == TACE_F64)
    return head_fwd<double>(x, row_of, w1, w2, n_nodes, channels, attrs, n_species, e0, scale, shift, batch, ptr,
                            rowptr, n_graphs, hid, vals, factor, node_energy, energy, s);
  return tace_fail_msg("tace_energy_head_fwd: dtype must be TACE_F32 or TACE_F64");
}

extern "C" int tace_energy_head_bwd(int dtype, const void* hid, const void* factor, const void* g_energy,
                                    const void* g_node, const int64_t* row_of, const int64_t* batch, const void* w1,
                                    int64_t n_nodes, int32_t channels, void* g_x, void* stream) {
  if (n_nodes < 0 || n_nodes > ((int64_t)1 << 31) || channels <= 0 || channels > HEAD_MAXC)
    return tace_fail_msg("tace_energy_head_bwd: bad sizes (1..512 channels)");
  if (n_nodes == 0) return 0;
  if (!hid || !factor || !row_of || !batch || !w1 || !g_x) return tace_fail_msg("tace_energy_head_bwd: null pointer");
  hipStream_t s = (hipStream_t)stream;
  if (dtype == TACE_F32)
    return head_bwd<float>(hid, factor, g_energy, g_node, row_of, batch, w1, n_nodes, channels, g_x, s);
  if (dtype == TACE_F64)
    return head_bwd<double>(hid, factor, g_energy, g_node, row_of, batch, w1, n_nodes, channels, g_x, s);
  return tace_fail_msg("tace_energy_head_bwd: dtype must be TACE_F32 or TACE_F64");
}
