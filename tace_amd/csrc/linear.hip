// MI355X (gfx950) segmented GEMM of the per-species linears
// (e3nnElementLinear, tace/models/linear.py:377-482: one o3.Linear weight per
// chemical element, applied to the nodes of that element).  On species-sorted,
// group-major node features a per-species linear is, per instruction and
// species, one [(rows of that species) x mul_in] @ [mul_in x mul_out] GEMM.
// With tens of species these GEMMs are tiny and one library launch each costs
// more than its arithmetic; this kernel runs ALL of them -- every output
// block, species and instruction of one linear -- in one launch.
//
// Work is described by a host-built table of square output tiles (edge 128:
// the float32 MFMA kernel, edge 64: the FMA kernel, float32 or float64).  A tile
// lies inside one output block and one species' row range, so one weight
// matrix per contributing instruction serves all its rows.  Per tile (8 x
// int64): out_base (element offset of the tile's first row in y), rows (<= edge),
// n (the block's width = row stride), c0 (first column), bias_off (element
// offset into bias, -1 = none), [cb, ce) (its contributions), unused.  Per
// contribution (4 x int64 + one double scale): x_base (element offset of the
// tile's first row in x), k (width of that input block = row stride), w_off
// (element offset of its weight matrix), trans (0: B = W [k, n] row-major;
// 1: B = W^T with W [n, k] row-major -- the input-gradient direction).
// Output: y[tile] = addend[tile] + alpha * (sum_c scale_c x_c[tile rows] @ B_c
// + bias), every element of every tile written once.  addend is optional (null:
// no term) and may be y itself (y += ...): each element is read before it is
// written, by the lane that writes it.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include "../../include/tace_hip.h"
#include "bf16x3.h"

int tace_fail_msg(const char* msg);   // tace_hip.hip
int tace_check_launch(const char* what);

namespace {

constexpr int TM = 64, TN = 64, TK = 16, PAD = 4;

// 256 threads = 16 x 16; thread (ty, tx) owns rows ty*4..ty*4+3 and columns
// tx*4..tx*4+3 of the tile.  A and B stage through LDS k-major (As[k][row],
// Bs[k][col]) so the inner product reads one 4-vector of each per k.
template <typename T>
__global__ __launch_bounds__(256) void k_seg_linear(const T* __restrict__ x, T* y, const T* addend,
                                                    const T* __restrict__ w, const T* __restrict__ bias,
                                                    const int64_t* __restrict__ tiles,
                                                    const int64_t* __restrict__ contribs,
                                                    const double* __restrict__ scales, T alpha) {
  __shared__ T As[TK][TM + PAD];
  __shared__ T Bs[TK][TN + PAD];
  const int64_t* td = tiles + 8 * (int64_t)blockIdx.x;
  const int64_t out_base = td[0];
  const int rows = (int)td[1], n = (int)td[2], c0 = (int)td[3];
  const int64_t bias_off = td[4];
  const int cb = (int)td[5], ce = (int)td[6];
  const int t = (int)threadIdx.x, tx = t & 15, ty = t >> 4;
  T acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = T(0);

  for (int c = cb; c < ce; ++c) {
    const int64_t* cd = contribs + 4 * (int64_t)c;
    const T* __restrict__ xa = x + cd[0];
    const int k = (int)cd[1];
    const T* __restrict__ wb = w + cd[2];
    const bool trans = cd[3] != 0;
    const T sc = (T)scales[c];
    for (int k0 = 0; k0 < k; k0 += TK) {
      // A: 64 rows x 16 k, consecutive threads along k (coalesced rows)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int r = (t >> 4) + 16 * p, kk = t & 15;
        As[kk][r] = (r < rows && k0 + kk < k) ? xa[(int64_t)r * k + k0 + kk] : T(0);
      }
      if (!trans) {
        // B[kk][col] = W[k0+kk][c0+col], consecutive threads along the column
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int kk = (t >> 6) + 4 * p, col = t & 63;
          Bs[kk][col] = (k0 + kk < k && c0 + col < n) ? sc * wb[(int64_t)(k0 + kk) * n + c0 + col] : T(0);
        }
      } else {
        // B[kk][col] = W[c0+col][k0+kk], consecutive threads along k
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int col = (t >> 4) + 16 * p, kk = t & 15;
          Bs[kk][col] = (k0 + kk < k && c0 + col < n) ? sc * wb[(int64_t)(c0 + col) * k + k0 + kk] : T(0);
        }
      }
      __syncthreads();
#pragma unroll
      for (int kk = 0; kk < TK; ++kk) {
        T a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
      }
      __syncthreads();
    }
  }
  T bv[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int col = c0 + tx * 4 + j;
    bv[j] = (bias_off >= 0 && col < n) ? bias[bias_off + col] : T(0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = ty * 4 + i;
    if (r >= rows) break;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = c0 + tx * 4 + j;
      if (col >= n) continue;
      const int64_t o = out_base + (int64_t)r * n + col;
      y[o] = alpha * (acc[i][j] + bv[j]) + (addend ? addend[o] : T(0));
    }
  }
}

// Global loads of the float32 MFMA path (k_seg_linear_bf16x3 below): every
// load is a 16-byte load, and the next 32-k chunk's loads are issued before
// the current chunk's MFMAs, so memory latency overlaps the matrix work.
typedef float f4 __attribute__((ext_vector_type(4)));

// one 16-byte load of p[0..3], or the first lim (< 4) elements and zeros
__device__ __forceinline__ f4 seg_ld4(const float* p, bool vec, bool any, int lim) {
  if (vec) return *(const f4*)p;
  f4 v = f4{0.f, 0.f, 0.f, 0.f};
  if (any) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < lim) v[e] = p[e];
  }
  return v;
}

// The MFMA kernels start each output's sum from addend / alpha (so that
// alpha (sum + bias) = addend + alpha (products + bias) up to rounding): the
// addend is read into the accumulators before the first MFMA, its loads in
// flight with the tile's first operand loads, instead of a load-add-store
// round trip per output row in the epilogue.  Rows past `rows` and columns
// past `ce` start from zero (they are not stored).
__device__ __forceinline__ f4 addend_init(const float* __restrict__ a, int64_t o, bool rok, int col, int ce,
                                          bool vec, float inv_alpha) {
  f4 v = f4{0.f, 0.f, 0.f, 0.f};
  if (rok) {
    if (vec && col + 4 <= ce) {
      v = *(const f4*)(a + o);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (col + q < ce) v[q] = a[o + q];
    }
  }
  return inv_alpha == 1.f ? v : v * inv_alpha;
}

// R rows x 32 k of a k-contiguous matrix (row stride k, `nrows` valid rows):
// thread t holds rows t/2 + 128 rr (rr < R/128), k k0 + 16 (t&1) .. +15 --
// one base address per row, four 16-byte loads at constant offsets
template <int R>
__device__ __forceinline__ void seg_load_k(const float* __restrict__ base, int k, int k0, int nrows, bool vec, int t,
                                           f4* v) {
  const int kk = k0 + 16 * (t & 1);
#pragma unroll
  for (int rr = 0; rr < R / 128; ++rr) {
    const int r = (t >> 1) + 128 * rr;
    const float* p = base + (int64_t)r * k + kk;
    const bool ok = r < nrows;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int left = k - (kk + 4 * q);
      v[4 * rr + q] = seg_ld4(p + 4 * q, ok && vec && left >= 4, ok && left > 0, left);
    }
  }
}

// float32 as three bfloat16 terms on the bf16 MFMA (v_mfma_f32_16x16x32_bf16,
// 2.3 PFLOP/s against 0.15 for the float32 MFMA): both operands split into
// three bf16 terms, six products per pair (bf16x3.h: the split is exact and
// the sums carry the rounding of a float32 GEMM).
//
// A tile is 128 x 128: 4 waves in a 2 x 2 grid, each owning 4 x 4 blocks of
// 16 x 16.  Tiles are taken XCD-grouped: workgroup b runs tile (b % 8) * per
// + b / 8, so XCD k works through a contiguous stretch of the table (the
// column tiles of one row tile, the row tiles of one species' weight) and
// shares them in its L2.  The split happens once per element at the LDS
// store, into three planes stored k-contiguous (rows of 32 k + 8 pad:
// 80-byte rows, so the 16 rows of a fragment read fall on distinct banks),
// and an MFMA fragment (8 k of one row) is one 16-byte LDS read.  The
// forward's W [k, n] is loaded two k rows per thread and stored transposed as
// (k, k + 1) pairs.
constexpr int SB_K = 32, SB_STR = SB_K + 8;
// rows of 16 k (four f4 of one row, k-contiguous) -> planes p[row][kofs ..]
template <bool SCALED>
__device__ __forceinline__ void sb_store_k16(unsigned short* lds, int plane, int off, const f4* v, float sc) {
  typedef unsigned u4v __attribute__((ext_vector_type(4)));
  u4v o[3][2];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      unsigned h[3];
      const bx3_f2 u = bx3_f2{v[q][2 * e], v[q][2 * e + 1]};
      bx3_split2(SCALED ? bx3_scale2(u, sc) : u, h);
#pragma unroll
      for (int p = 0; p < 3; ++p) o[p][q >> 1][2 * (q & 1) + e] = h[p];
    }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    *(u4v*)&lds[p * plane + off] = o[p][0];
    *(u4v*)&lds[p * plane + off + 8] = o[p][1];
  }
}

// 8 k of one row (two f4, k-contiguous) -> planes p[row][kofs ..]
__device__ __forceinline__ void sb_store_k8(unsigned short* lds, int plane, int off, const f4 (&v)[2]) {
  const float u[8] = {v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
  bx3_bf8 h[3];
  bx3_split8(u, h);
#pragma unroll
  for (int p = 0; p < 3; ++p) *(bx3_bf8*)&lds[p * plane + off] = h[p];
}

// 32 k rows x 128 columns of W [k, n] from column c0: thread t holds k rows
// k0 + 2 (t/16) and the next, columns 4 (t%16) + 64 q (q < 2) -- v[2 q + r]
// for row 2 (t/16) + r
__device__ __forceinline__ void sb_load_n(const float* __restrict__ wb, int k, int n, int c0, int k0, bool vec, int t,
                                          f4* v) {
  const int cb = c0 + 4 * (t & 15);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int kk = k0 + 2 * (t >> 4) + r;
    const float* p = wb + (int64_t)kk * n + cb;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int left = n - (cb + 64 * q);
      v[2 * q + r] = seg_ld4(p + 64 * q, kk < k && vec && left >= 4, kk < k && left > 0, left);
    }
  }
}

// Lane t writes its four columns 4 (t%16) + e in the order e = (e' + r) & 3,
// r = (t/4) & 3, so that a store instruction (fixed e') spreads the 16 lanes
// of a row group over distinct banks instead of four.
__device__ __forceinline__ void sb_store_n(unsigned short* lds, int plane, int t, const f4* v, float sc) {
  const int kp = 2 * (t >> 4), r = (t >> 2) & 3;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    f4 u0, u1;   // v rotated left by r
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f4 x0 = v[2 * q], x1 = v[2 * q + 1];
      u0[e] = r == 0 ? x0[e] : r == 1 ? x0[(e + 1) & 3] : r == 2 ? x0[(e + 2) & 3] : x0[(e + 3) & 3];
      u1[e] = r == 0 ? x1[e] : r == 1 ? x1[(e + 1) & 3] : r == 2 ? x1[(e + 2) & 3] : x1[(e + 3) & 3];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      unsigned h[3];   // (k, k + 1) of one column
      bx3_split2(bx3_scale2(bx3_f2{u0[e], u1[e]}, sc), h);
      const int col = 4 * (t & 15) + 64 * q + ((e + r) & 3);
#pragma unroll
      for (int p = 0; p < 3; ++p) *(unsigned*)&lds[p * plane + col * SB_STR + kp] = h[p];
    }
  }
}

__global__ __launch_bounds__(256) void k_seg_linear_bf16x3(const float* __restrict__ x, float* y,
                                                           const float* addend, const float* __restrict__ w,
                                                           const float* __restrict__ bias,
                                                           const int64_t* __restrict__ tiles,
                                                           const int64_t* __restrict__ contribs,
                                                           const double* __restrict__ scales, float alpha,
                                                           int n_tiles, int per) {
  constexpr int WM = 4, WN = 4, TR = 128, TC = 128, PL = 128 * SB_STR;   // plane size (bf16)
  __shared__ __attribute__((aligned(16))) unsigned short As[3 * PL];
  __shared__ __attribute__((aligned(16))) unsigned short Bs[3 * PL];
  const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tile >= n_tiles) return;
  const int64_t* td = tiles + 8 * (int64_t)tile;
  const int64_t out_base = td[0];
  const int rows = (int)td[1], n = (int)td[2], c0 = (int)td[3];
  const int64_t bias_off = td[4];
  const int cb = (int)td[5], ce = (int)td[6];
  const int t = (int)threadIdx.x, lane = t & 63, wv = t >> 6;
  const int wr = (wv >> 1) * 16 * WM, wc = (wv & 1) * 16 * WN;
  const int fr = lane & 15, fg = lane >> 4;
  f4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  const int soff = (t >> 1) * SB_STR + 16 * (t & 1);   // this thread's k16 run of a k-contiguous plane

  for (int c = cb; c < ce; ++c) {
    const int64_t* cd = contribs + 4 * (int64_t)c;
    const float* __restrict__ xa = x + cd[0];
    const int k = (int)cd[1];
    const float* __restrict__ wb = w + cd[2];
    const bool trans = cd[3] != 0;
    const float sc = (float)scales[c];
    const bool xvec = ((((uintptr_t)xa) & 15) == 0) && ((k & 3) == 0);
    const bool wvec = ((((uintptr_t)wb) & 15) == 0) && (((trans ? k : n) & 3) == 0) && ((c0 & 3) == 0);
    const float* __restrict__ wt = wb + (int64_t)c0 * k;
    f4 a[4], b[4];
    auto load = [&](int kc, f4* a, f4* b) {
      seg_load_k<TR>(xa, k, kc, rows, xvec, t, a);
      if (trans) seg_load_k<TC>(wt, k, kc, n - c0, wvec, t, b);
      else sb_load_n(wb, k, n, c0, kc, wvec, t, b);
    };
    auto stage = [&](const f4* a, const f4* b) {
      sb_store_k16<false>(As, PL, soff, a, 1.f);
      if (trans) sb_store_k16<true>(Bs, PL, soff, b, sc);
      else sb_store_n(Bs, PL, t, b, sc);
    };
    auto mma = [&]() {
      bx3_bf8 af[3][WM];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int i = 0; i < WM; ++i) af[p][i] = *(const bx3_bf8*)&As[p * PL + (wr + 16 * i + fr) * SB_STR + 8 * fg];
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        bx3_bf8 bf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) bf[p] = *(const bx3_bf8*)&Bs[p * PL + (wc + 16 * j + fr) * SB_STR + 8 * fg];
#pragma unroll
        for (int u = 0; u < 6; ++u)   // the six terms a_i b_j, smallest first
#pragma unroll
          for (int i = 0; i < WM; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[BX3_TA[u]][i], bf[BX3_TB[u]], acc[i][j], 0, 0, 0);
      }
    };
    load(0, a, b);
    for (int k0 = 0; k0 < k; k0 += SB_K) {
      stage(a, b);
      __syncthreads();
      if (k0 + SB_K < k) load(k0 + SB_K, a, b);   // next chunk in flight during this chunk's MFMAs
      mma();
      __syncthreads();
    }
  }
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int col = c0 + wc + 16 * j + fr;
    if (col >= n) continue;
    const float bv = bias_off >= 0 ? bias[bias_off + col] : 0.f;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = wr + 16 * i + 4 * fg + q;
        if (r >= rows) continue;
        const int64_t o = out_base + (int64_t)r * n + col;
        y[o] = alpha * (acc[i][j][q] + bv) + (addend ? addend[o] : 0.f);
      }
  }
}

// ---- the same GEMM with the weights split ahead of time ------------------
// The weights of the per-species linears are constants at inference, so their
// three bf16 terms (with the contribution's scale folded in) are made once,
// by k_split_blocks, into three planes laid out the way the LDS tile holds
// them: per weight block, column-major runs of k_pad = ceil8(k) bf16 (zeros
// past k), column c of the block at w_off + c k_pad of each plane.  The GEMM
// then stages B with plain 16-byte copies -- no split, no transposition, no
// scale -- which removes most of the kernel's VALU work and the transposed
// LDS stores.

// 128 columns x 32 k of one contribution's B: thread t stages column t / 2,
// k k0 + 16 (t & 1) .. + 15, of each plane (two 16-byte loads per plane; a
// k_pad run is a multiple of 8, so each load is wholly inside or outside it)
typedef unsigned u4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void sbs_load(const unsigned short* __restrict__ wp, int64_t pstride, int kpad, int ncols,
                                         int k0, int t, u4v* v) {
  const int col = t >> 1, kk = k0 + 16 * (t & 1);
  const unsigned short* p = wp + (int64_t)col * kpad + kk;
#pragma unroll
  for (int pl = 0; pl < 3; ++pl)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool ok = col < ncols && kk + 8 * h < kpad;
      v[2 * pl + h] = ok ? *(const u4v*)(p + pl * pstride + 8 * h) : u4v{0u, 0u, 0u, 0u};
    }
}

__device__ __forceinline__ void sbs_store(unsigned short* lds, int plane, int off, const u4v* v) {
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) {
    *(u4v*)&lds[pl * plane + off] = v[2 * pl];
    *(u4v*)&lds[pl * plane + off + 8] = v[2 * pl + 1];
  }
}

__global__ __launch_bounds__(256) void k_seg_linear_bx3s(const float* __restrict__ x, float* y, const float* addend,
                                                         const unsigned short* __restrict__ wsp, int64_t pstride,
                                                         const float* __restrict__ bias,
                                                         const int64_t* __restrict__ tiles,
                                                         const int64_t* __restrict__ contribs, float alpha,
                                                         int n_tiles, int per) {
  constexpr int WM = 4, WN = 4, TR = 128, PL = 128 * SB_STR;   // plane size (bf16)
  __shared__ __attribute__((aligned(16))) unsigned short As[3 * PL];
  __shared__ __attribute__((aligned(16))) unsigned short Bs[3 * PL];
  const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tile >= n_tiles) return;
  const int64_t* td = tiles + 8 * (int64_t)tile;
  const int64_t out_base = td[0];
  const int rows = (int)td[1], n = (int)td[2], c0 = (int)td[3];
  const int64_t bias_off = td[4];
  const int cb = (int)td[5], ce = (int)td[6];
  const int t = (int)threadIdx.x, lane = t & 63, wv = t >> 6;
  const int wr = (wv >> 1) * 16 * WM, wc = (wv & 1) * 16 * WN;
  const int fr = lane & 15, fg = lane >> 4;
  f4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  const int soff = (t >> 1) * SB_STR + 16 * (t & 1);   // this thread's k16 run of a k-contiguous plane

  for (int c = cb; c < ce; ++c) {
    const int64_t* cd = contribs + 4 * (int64_t)c;
    const float* __restrict__ xa = x + cd[0];
    const int k = (int)cd[1];
    const int kpad = (k + 7) & ~7;
    const unsigned short* __restrict__ wp = wsp + cd[2] + (int64_t)c0 * kpad;
    const bool xvec = ((((uintptr_t)xa) & 15) == 0) && ((k & 3) == 0);
    f4 a[4];
    u4v b[6];
    auto load = [&](int kc) {
      seg_load_k<TR>(xa, k, kc, rows, xvec, t, a);
      sbs_load(wp, pstride, kpad, n - c0, kc, t, b);
    };
    auto mma = [&]() {
      bx3_bf8 af[3][WM];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int i = 0; i < WM; ++i) af[p][i] = *(const bx3_bf8*)&As[p * PL + (wr + 16 * i + fr) * SB_STR + 8 * fg];
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        bx3_bf8 bf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) bf[p] = *(const bx3_bf8*)&Bs[p * PL + (wc + 16 * j + fr) * SB_STR + 8 * fg];
#pragma unroll
        for (int u = 0; u < 6; ++u)   // the six terms a_i b_j, smallest first
#pragma unroll
          for (int i = 0; i < WM; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[BX3_TA[u]][i], bf[BX3_TB[u]], acc[i][j], 0, 0, 0);
      }
    };
    load(0);
    for (int k0 = 0; k0 < k; k0 += SB_K) {
      sb_store_k16<false>(As, PL, soff, a, 1.f);
      sbs_store(Bs, PL, soff, b);
      __syncthreads();
      if (k0 + SB_K < k) load(k0 + SB_K);   // next chunk in flight during this chunk's MFMAs
      mma();
      __syncthreads();
    }
  }
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int col = c0 + wc + 16 * j + fr;
    if (col >= n) continue;
    const float bv = bias_off >= 0 ? bias[bias_off + col] : 0.f;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = wr + 16 * i + 4 * fg + q;
        if (r >= rows) continue;
        const int64_t o = out_base + (int64_t)r * n + col;
        y[o] = alpha * (acc[i][j][q] + bv) + (addend ? addend[o] : 0.f);
      }
  }
}

// ---- the tile kernel with B in fragment order ----------------------------
// k_seg_linear_bx3s stages A and B through LDS with two barriers per 32-k
// step; LDS traffic (48 KB of plane stores and 96 KB of fragment reads per
// step and workgroup) then takes about as long as the MFMAs.  Here:
//  * B fragments come straight from the weights pre-split in MFMA fragment
//    order (k_split_blocks layout 1, as the task kernel reads them): one
//    coalesced 16-byte load per lane and fragment, one step ahead;
//  * A (128 rows x 32 k) is loaded two steps ahead and split into the three
//    planes in LDS, double buffered: step s + 1's planes are written after
//    step s's MFMAs, and one barrier per step separates them;
//  * every load is unconditional (past the last step it repeats that step):
//    a load under a branch makes the compiler wait for all loads at the
//    join, the prefetches included;
//  * the MFMA runs with the operands swapped (B fragments as the row
//    operand), so a lane holds 4 consecutive columns of one output row, and
//    the stores trade blocks between lanes fr and fr ^ 8 as the task kernel's
//    do (8 whole rows of 32 columns per store).
//  * a workgroup takes 64 of the tile's 128 rows, each wavefront all of them
//    for 32 columns: 142 registers, so three workgroups run per CU and one's
//    MFMAs cover another's loads and splits (a whole tile per workgroup, 2 x 2
//    wavefronts of 64 x 64, ran two at 232 registers), and row blocks past
//    the tile's rows are left out 32 at a time.  Taller or wider wavefront
//    tiles (128 x 32 with two workgroups per CU) measured slower.  The tables'
//    XCD runs matter as much (_xcd_balanced in ops.py).  Both together, whole
//    tiles in runs of equal length -> halves in runs of equal cost: 12,288
//    rows x (1 + 3 + 5 + 7), k 2,944-5,376 into 128 columns, 1660 -> 1325 us
//    (143 -> 179 TFLOP/s, 3.50 -> 2.46 M cycles, MFMA pipe 39 -> 56% busy); the
//    same at 1,024 rows and 4 species 167 -> 145 us; 128 -> 128 shared linears
//    52 -> 51 us.  Part of what is left is power: 1,164 us with all operands
//    zero, and a library bf16 product goes from 1,337 TFLOP/s on random
//    operands to 1,707 on zeros.
// Tiles, contributions and the XCD-grouped tile order are those of
// k_seg_linear_bx3s (entries of 0 rows are skipped); contribution column 2 is
// the block's offset in the fragment-order weights.  Per output element the products and their order
// are those of k_seg_linear_bx3s (contributions and k steps in order, the six
// terms smallest first, each a sum over the same 32 products), so the two
// kernels give the same bits.
struct FtLoad {   // the contribution and step whose operands load next
  const float* xa;
  const unsigned short* wf;
  int c, s, k, nks, send;   // steps s .. send - 1 of the contribution's nks
  bool xvec;
};

struct FtDense {   // the sizes of a launch without tables: one [m, k] x [k, n] product
  int64_t m;
  int n, k;
};

__device__ __forceinline__ void ft_open(FtLoad& L, const float* __restrict__ x, const unsigned short* __restrict__ wfrag,
                                        const int64_t* __restrict__ contribs, int c, const FtDense& dense) {
  const int64_t* cd = contribs + 4 * (int64_t)c;
  L.c = c;
  L.s = 0;
  L.xa = contribs ? x + cd[0] : x;
  L.k = contribs ? (int)cd[1] : dense.k;
  L.nks = (L.k + 31) >> 5;
  L.send = L.nks;
  L.wf = contribs ? wfrag + cd[2] : wfrag;
  L.xvec = ((((uintptr_t)L.xa) & 15) == 0) && ((L.k & 3) == 0);
}

// A (64 rows from r0 x 32 k) of step L.s: thread t holds row t / 4, k 8 (t & 3)
// .. + 7.  Rows past nrows repeat the last row (their outputs are not stored).
// VEC (every contribution 16-byte aligned with k % 4 == 0): two unconditional
// 16-byte loads, a run past k read from the row's start and zeroed -- no branch, so
// the compiler's wait for this step's B (issued before) is exact.
template <bool VEC>
__device__ __forceinline__ void ft_load_a(const FtLoad& L, int r0, int nrows, int t, f4 (&v)[2]) {
  const int kk = 32 * L.s + 8 * (t & 3);
  const int r = r0 + min(t >> 2, nrows - 1);
  const float* row = L.xa + (int64_t)r * L.k;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int left = L.k - (kk + 4 * q);
    if constexpr (VEC) {
      const f4 u = *(const f4*)(left >= 4 ? row + kk + 4 * q : row);
      v[q] = left >= 4 ? u : f4{0.f, 0.f, 0.f, 0.f};
    } else {
      v[q] = seg_ld4(row + kk + 4 * q, false, left > 0, left);
    }
  }
}

// B fragments (three terms) of column blocks jb0 and jb0 + 1 (clamped to the
// block's last) at step L.s
__device__ __forceinline__ void ft_load_b(const FtLoad& L, int jb0, int nb16, int lane, u4v (&d)[3][2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int jb = min(jb0 + j, nb16 - 1);
    const unsigned short* p = L.wf + ((int64_t)(jb * L.nks + L.s) * 3) * 512 + 8 * lane;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) d[pl][j] = *(const u4v*)(p + pl * 512);
  }
}

//
// SPLIT (split k, for launches with too few tiles to fill the chip, or long k
// over more weights than the caches hold): item vi = tile * splits + sp sums steps [sp nks / splits, (sp + 1) nks /
// splits) of the tile's first contribution into its own 128 x 128 partial
// tile, partials + 16384 vi (row stride 128), with no addend, bias or alpha;
// k_seg_split_sum adds the partials up (NaN for a tile with more than one
// contribution).
template <bool VEC, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_seg_linear_bx3f(
    const float* __restrict__ x, float* y, const float* addend, const unsigned short* __restrict__ wfrag,
    const float* __restrict__ bias, const int64_t* __restrict__ tiles, const int64_t* __restrict__ contribs,
    float alpha, int n_tiles, int per, int splits, float* __restrict__ partials, FtDense dense) {
  constexpr int WM = 4, PL = 64 * SB_STR;   // 16-row blocks, plane size (bf16)
  __shared__ __attribute__((aligned(16))) unsigned short As[2][3 * PL];
  // work item wi: split sp of a tile, half of its rows.  The two halves run
  // next to each other on one XCD, and all tiles' first k range comes before
  // their second: tiles that read the same weights start within a few steps
  // of each other, so what one of them loads the others find in L2.  (With
  // the splits of a tile side by side, or unsplit, the row tiles of a long-k
  // block drift apart by more steps than L2 holds: 5,003 rows of 89 species,
  // k 5,888-10,752 into 256 columns, 4.8 GB of weights: 20.7 GB read and 3,451
  // us unsplit, 3,281 us in 4 neighbouring splits, 16.3 GB and 2,710 us this way.)
  const int half = (int)(blockIdx.x >> 3) & 1;
  const int wi = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 4);
  const int sp = SPLIT ? wi / n_tiles : 0, tile = SPLIT ? wi - sp * n_tiles : wi;
  const int vi = SPLIT ? tile * splits + sp : tile;
  if (SPLIT ? sp >= splits : tile >= n_tiles) return;
  const int64_t* td = tiles + 8 * (int64_t)tile;
  const int r0 = 64 * half;
  int rows, n, c0, cb = 0, ce = 1;
  int64_t out_base, bias_off = -1;
  if (tiles) {
    rows = min((int)td[1] - r0, 64);
    n = (int)td[2];
    c0 = (int)td[3];
    out_base = td[0] + (int64_t)r0 * n;
    if constexpr (!SPLIT) bias_off = td[4];
    cb = (int)td[5];
    ce = (int)td[6];
  } else {
    // one [m, k] x [k, n] product: the column tiles of a row tile in turn
    const int ct = (dense.n + 127) >> 7, rt = tile / ct;
    rows = (int)min(dense.m - 128 * (int64_t)rt - r0, (int64_t)64);
    n = dense.n;
    c0 = 128 * (tile - rt * ct);
    out_base = (128 * (int64_t)rt + r0) * n;
    if (bias) bias_off = 0;
    x += 128 * (int64_t)rt * dense.k;
  }
  if (rows <= 0) return;   // the tile ends in the first half, or a padding entry of the table
  if constexpr (SPLIT) ce = min(ce, cb + 1);   // k_seg_split_sum writes NaN for a tile with more
  const int t = (int)threadIdx.x, lane = t & 63, wv = t >> 6;
  const int wc = wv * 32;   // this wavefront's 32 columns (all 64 rows)
  const int fr = lane & 15, fg = lane >> 4;
  const int nb16 = (n + 15) >> 4, jb0 = (c0 + wc) >> 4;
  const int soff = (t >> 2) * SB_STR + 8 * (t & 3);   // this thread's 8 k of a k-contiguous plane

  f4 acc[WM][2];
  if (!SPLIT && addend) {
    const bool avec = ((n & 3) == 0) && ((out_base & 3) == 0) && ((((uintptr_t)addend) & 15) == 0);
    const float ia = 1.f / alpha;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = 16 * i + fr, col = c0 + wc + 16 * j + 4 * fg;
        acc[i][j] = addend_init(addend, out_base + (int64_t)r * n + col, r < rows, col, n, avec, ia);
      }
  } else {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  }

  // skip contributions without k steps
  int c = cb;
  FtLoad L;
  while (c < ce) {
    ft_open(L, x, wfrag, contribs, c, dense);
    if constexpr (SPLIT) {
      L.s = (int)((int64_t)sp * L.nks / splits);
      L.send = (int)((int64_t)(sp + 1) * L.nks / splits);
    }
    if (L.send > L.s) break;
    ++c;
  }
  if (c < ce) {
    // the steps of all contributions, in order.  A loads two steps ahead of
    // the MFMAs (cursor LA; A(j) in register set j & 1), B one step ahead
    // (cursor LB): x streams from HBM, the weights from L2
    FtLoad LA = L, LB = L;
    bool moreA = true, moreB = true;
    // C to the step after the one it names; after the last step C stays
    // there (more = false), so the loads below never need a condition
    auto advance = [&](FtLoad& C, bool& more) {
      if (C.s + 1 < C.send) {
        ++C.s;
        return;
      }
      if constexpr (SPLIT) {   // one contribution
        more = false;
        return;
      }
      for (int cc = C.c + 1; cc < ce; ++cc) {
        FtLoad D;
        ft_open(D, x, wfrag, contribs, cc, dense);
        if (D.send > 0) {
          C = D;
          return;
        }
      }
      more = false;
    };
    f4 a0[2], a1[2];
    u4v b0[3][2], b1[3][2];
    ft_load_a<VEC>(LA, r0, rows, t, a0);
    advance(LA, moreA);
    ft_load_b(LB, jb0, nb16, lane, b0);
    advance(LB, moreB);
    ft_load_a<VEC>(LA, r0, rows, t, a1);   // (a repeat of the last step when there is no next)
    advance(LA, moreA);
    sb_store_k8(As[0], PL, soff, a0);
    __syncthreads();
    // step g: MFMAs on LDS buffer `buf` (= g & 1) and fragments cur while A(g
    // + 2) loads into al and B(g + 1) into nxt; then A(g + 1) (in as) split
    // into the other buffer
    auto step = [&](int buf, const u4v (&cur)[3][2], u4v (&nxt)[3][2], f4 (&al)[2], const f4 (&as)[2]) {
      const bool have = moreB;
      // B before A: vector loads complete in issue order, so waiting for
      // this step's B (issued last step) does not wait for the A issued
      // after it.  Unconditional (repeats past the last step): a load under
      // a branch makes the compiler wait for every load at the join
      ft_load_b(LB, jb0, nb16, lane, nxt);
      advance(LB, moreB);
      ft_load_a<VEC>(LA, r0, rows, t, al);
      advance(LA, moreA);
      __builtin_amdgcn_sched_barrier(0);
      const unsigned short* Ab = As[buf];
#pragma unroll
      for (int ip = 0; ip < WM / 2; ++ip) {
        if (ip > 0 && rows <= 32 * ip) break;   // no such rows (uniform)
        bx3_bf8 af[2][3];
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
          for (int pl = 0; pl < 3; ++pl)
            af[ii][pl] = *(const bx3_bf8*)&Ab[pl * PL + (32 * ip + 16 * ii + fr) * SB_STR + 8 * fg];
#pragma unroll
        for (int u = 0; u < 6; ++u)   // the six terms a_i b_j, smallest first
#pragma unroll
          for (int ii = 0; ii < 2; ++ii)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[2 * ip + ii][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  __builtin_bit_cast(bx3_bf8, cur[BX3_TB[u]][j]), af[ii][BX3_TA[u]], acc[2 * ip + ii][j], 0, 0, 0);
      }
      // the next A's split after the MFMAs (interleaving it measured slower)
      __builtin_amdgcn_sched_barrier(0);
      sb_store_k8(As[buf ^ 1], PL, soff, as);
      __syncthreads();
      return have;
    };
    while (step(0, b0, b1, a0, a1) && step(1, b1, b0, a1, a0)) {
    }
  }

  // which of this lane's outputs are not finite (bit 8 i + 4 j + q); none in
  // all but rare tiles, so one sum of zeros asks first (a test of every output
  // cost 3% of a TECE layer's products)
  unsigned odd = 0;
  if constexpr (!SPLIT) {
    if (!tiles) {
      float z = 0.f;
#pragma unroll
      for (int e = 0; e < 8 * WM; ++e) z = fmaf(acc[e >> 3][(e >> 2) & 1][e & 3], 0.f, z);
      if (z != z) {
#pragma unroll
        for (int e = 0; e < 8 * WM; ++e) odd |= (unsigned)!__builtin_isfinite(acc[e >> 3][(e >> 2) & 1][e & 3]) << e;
      }
    }
  }
  // the bias of this lane's 8 columns (no loads are outstanding here)
  f4 bv[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    bv[j] = f4{0.f, 0.f, 0.f, 0.f};
    if (bias_off >= 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) bv[j][q] = bias[bias_off + min(c0 + wc + 16 * j + 4 * fg + q, n - 1)];
    }
  }
  // acc[i][j][q] = out[row 16 i + fr][column c0 + wc + 16 j + 4 fg + q];
  // lanes fr and fr ^ 8 trade one block, so a store writes 8 whole rows of 32 columns
  const bool vst = SPLIT || (((n & 3) == 0) && ((out_base & 3) == 0) && ((((uintptr_t)y) & 15) == 0));
  const float osc = SPLIT ? 1.f : alpha;
  const bool lo = fr < 8;
  const int jl = lo ? 0 : 1;
  const int col = c0 + wc + 16 * jl + 4 * fg;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const f4 v0 = osc * (acc[i][0] + bv[0]), v1 = osc * (acc[i][1] + bv[1]);
    const f4 give = lo ? v1 : v0;
    f4 got;
#pragma unroll
    for (int q = 0; q < 4; ++q) got[q] = __shfl_xor(give[q], 8);
    const f4 s0 = lo ? v0 : got, s1 = lo ? got : v1;   // rows 16 i + (fr & 7), + 8
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = 16 * i + 8 * h + (fr & 7);
      if (r >= rows || col >= n) continue;
      const f4 v = h ? s1 : s0;
      float* dst = SPLIT ? partials + 16384 * (int64_t)vi + 128 * (r0 + r) + (col - c0)
                         : y + out_base + (int64_t)r * n + col;
      if (vst) {
        *(f4*)dst = v;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (col + q < n) dst[q] = v[q];
      }
    }
  }
  if constexpr (!SPLIT) {
    // The dense product has the infinities of a float32 one: an infinity, or an
    // x past bf16's largest, splits into terms of both signs, so its outputs
    // came out NaN.  They are summed once more in order (rare; a sum that is
    // NaN ends there).
    if (odd) {
      __threadfence_block();   // behind the other lanes' stores of the same outputs
      const int nks = (dense.k + 31) >> 5;
      for (; odd; odd &= odd - 1) {
        const int e = __ffs(odd) - 1, r = 16 * (e >> 3) + fr, cl = c0 + wc + 16 * ((e >> 2) & 1) + 4 * fg + (e & 3);
        if (r >= rows || cl >= n) continue;
        const float* xr = x + (int64_t)(r0 + r) * dense.k;
        const unsigned short* wc0 = wfrag + (int64_t)(cl >> 4) * nks * 1536 + 8 * (cl & 15);
        float s = 0.f;
        for (int kk = 0; kk < dense.k && s == s; ++kk) {
          const unsigned short* w = wc0 + (int64_t)(kk >> 5) * 1536 + 128 * ((kk & 31) >> 3) + (kk & 7);
          const float w0 = __uint_as_float((unsigned)w[0] << 16);
          const float wv = __builtin_isinf(w0)
              ? w0 : w0 + (__uint_as_float((unsigned)w[512] << 16) + __uint_as_float((unsigned)w[1024] << 16));
          s = fmaf(xr[kk], wv, s);
        }
        y[out_base + (int64_t)r * n + cl] = bias ? s + bias[cl] : s;
      }
    }
  }
}

// The partial tiles of k_seg_linear_bx3f<*, true> added up, 16 workgroups
// per tile (8 rows each, a thread per 4 columns of a row): y = alpha
// (addend / alpha + partial_0 + ... + partial_{splits-1} + bias), the partials
// in split order (a fixed order, so every run gives the same bits); NaN in
// every output of a tile with more than one contribution (the split kernel
// sums only its first).  The addend may be y itself: each element is read
// and then written by the same thread.
__global__ __launch_bounds__(256) void k_seg_split_sum(float* y, const float* addend, const float* __restrict__ bias,
                                                       const int64_t* __restrict__ tiles,
                                                       const float* __restrict__ partials, int splits, float alpha) {
  const int tile = (int)(blockIdx.x >> 4);
  const int64_t* td = tiles + 8 * (int64_t)tile;
  const int64_t out_base = td[0], bias_off = td[4];
  const int rows = (int)td[1], n = (int)td[2], c0 = (int)td[3];
  const int r = 8 * (int)(blockIdx.x & 15) + ((int)threadIdx.x >> 5), cc = 4 * ((int)threadIdx.x & 31), col = c0 + cc;
  if (r >= rows || col >= n) return;
  const bool bad = td[6] - td[5] > 1;
  const bool vec = ((n & 3) == 0) && ((out_base & 3) == 0) && ((((uintptr_t)y) & 15) == 0);
  const bool avec = vec && ((((uintptr_t)addend) & 15) == 0);
  const int64_t o = out_base + (int64_t)r * n + col;
  f4 acc = addend ? addend_init(addend, o, true, col, n, avec, 1.f / alpha) : f4{0.f, 0.f, 0.f, 0.f};
  const float* __restrict__ P = partials + (int64_t)tile * splits * 16384 + 128 * r + cc;
#pragma unroll 4
  for (int s = 0; s < splits; ++s) acc += *(const f4*)(P + (int64_t)s * 16384);
  f4 b = f4{0.f, 0.f, 0.f, 0.f};
  if (bias_off >= 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (col + q < n) b[q] = bias[bias_off + col + q];
  }
  const f4 out = bad ? f4{NAN, NAN, NAN, NAN} : alpha * (acc + b);
  if (vec && col + 4 <= n) {
    *(f4*)(y + o) = out;
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (col + q < n) y[o + q] = out[q];
  }
}

// ---- short k, wide n: the input-gradient shape ---------------------------
// The input gradients of the product-basis contractions are [rows, k = 128]
// x [128, n] with n up to ~5,400 columns per output block.  A 128 x 128 tile
// of the kernel above does four 32-k steps after staging A and B through LDS
// with two barriers per step, then writes its outputs one float per lane.
// Here a workgroup owns one R-row tile of one contribution with k <= KM
// and a range of columns:
//  * A is split once into the three bf16 planes in LDS (k-contiguous rows of
//    KM + 8 bf16, so the 16 rows of a fragment read fall on distinct banks),
//    its loads all in flight together; one barrier, none after it;
//  * GROUPS groups of four wavefronts take the range's 128-column tiles in
//    turn; a wavefront owns all R rows of 32 columns, so each B fragment
//    is loaded by one wavefront only; a tile of at most 32 rows (a species'
//    last one) multiplies two row blocks instead of four;
//  * B comes from weights pre-split in MFMA fragment order (k_split_blocks,
//    layout 1): the three terms of one 16-column x 32-k fragment are three
//    contiguous 1 KB runs in lane order, so a fragment is one fully
//    coalesced 16-byte load per lane.  Loaded one 32-k step ahead, and across
//    the end of a column tile: the next tile's first step is in flight before
//    this tile's stores, so no wait covers them.  The loads are unconditional
//    (the column block clamped into the weight block);
//  * the MFMA runs with the operands swapped (B fragments as the row operand),
//    so a lane holds 4 consecutive columns of one output row: one 16-byte
//    store per 16 x 16 block.
// The number of 32-k steps is a template parameter (1..KM / 32).  Per output element
// the products and their order are those of k_seg_linear_bx3s (k steps in
// order, the six terms smallest first, each a sum over the same 32 products),
// so the two kernels give the same bits.
//
// Task table (10 x int64): out_base (element offset of the tile's row 0,
// column 0 in y), rows (<= R), n (block width = row stride of y), [cb, ce)
// (the columns, ce <= n), bias_off (-1 none), x_base (element offset of the
// tile's row 0 in x), k (0..KM, the row stride of x; 0 = no contribution:
// the tile is alpha * bias or zero), w_off (the block's offset in the
// fragment-order weights), unused.
//
// Two shapes, both of 64 rows: k <= 128 in one group (52 KB of LDS, three
// workgroups per CU), k <= 256 in two groups (101 KB, one).  Large launches
// are bound by power and by the writes: 5,184 rows of the 593 x 128 columns of
// a product basis take 671 us, 442 in a copy without the stores (1.6 GB; the
// two add up) and 10% less with all operands zero; 709 us with 128 rows per
// workgroup and one workgroup per CU, whose operands came in and went out
// behind nothing.  Small ones gain from the
// smaller workgroups: 64 rows 41 -> 18 us, 400 rows 88 -> 55, 1,024 rows
// 170 -> 164, 3,000 rows of 89 species 584 -> 538.  For k <= 256, 32 rows in
// three workgroups per CU read B twice as often: 3,180 us became 3,431 (6,656
// rows, 89 species, 256 channels; 3,258 before the loads in flight and the
// plain stores).
template <int R_, int KM_, int GROUPS>
struct KsShape {
  static constexpr int R = R_, KM = KM_, RB = R / 16, STR = KM + 8, PL = R * STR;
  static constexpr int WAVES = GROUPS == 1 ? 3 : 2;   // wavefronts per SIMD
  static constexpr int THREADS = 256 * GROUPS, CSTEP = 128 * GROUPS;
};

struct KsTask {
  int64_t out_base, bias_off;
  int rows, n, cb, ce, nks, nb16;
  const unsigned short* wf;
  const float* addend;   // added to the outputs (null: none; may be y)
};

// B fragments (three terms, column blocks 2 wq and 2 wq + 1 of column tile c)
// of step ks into d; the column block clamped to the weight block's last
__device__ __forceinline__ void ks_load_b(const KsTask& T, int c, int ks, int wq, int lane, u4v (&d)[3][2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int jb = min((c >> 4) + 2 * wq + j, T.nb16 - 1);
    const unsigned short* p = T.wf + ((int64_t)(jb * T.nks + ks) * 3) * 512 + 8 * lane;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) d[pl][j] = *(const u4v*)(p + pl * 512);
  }
}

// step KS of a column tile: MFMAs on cur while the next step's fragments
// (or the next tile's first) load into nxt; RB: 16-row blocks that hold rows
template <class S, int RB, int NKS, int KS>
__device__ __forceinline__ void ks_step(const unsigned short* __restrict__ As, const KsTask& T, int c, int wq,
                                        int lane, int fr, int fg, f4 (&acc)[RB][2], const u4v (&cur)[3][2],
                                        u4v (&nxt)[3][2]) {
  if (KS + 1 < NKS) ks_load_b(T, c, KS + 1, wq, lane, nxt);
  else ks_load_b(T, c + S::CSTEP, 0, wq, lane, nxt);
  // the loads go out before this step's MFMAs (the scheduler would sink them
  // to the end of the step, where nothing hides their latency)
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ip = 0; ip < RB / 2; ++ip) {   // row blocks in pairs: four independent accumulators per term
    bx3_bf8 af[2][3];
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        af[ii][pl] = *(const bx3_bf8*)&As[pl * S::PL + (32 * ip + 16 * ii + fr) * S::STR + 32 * KS + 8 * fg];
#pragma unroll
    for (int u = 0; u < 6; ++u)   // the six terms a_i b_j, smallest first
#pragma unroll
      for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[2 * ip + ii][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bx3_bf8, cur[BX3_TB[u]][j]), af[ii][BX3_TA[u]], acc[2 * ip + ii][j], 0, 0, 0);
  }
  // keep the next step's LDS reads out of this one
  __builtin_amdgcn_sched_barrier(0);
}

// steps KS.. of a column tile; step KS reads buffer (KS + PAR) & 1
template <class S, int RB, int NKS, int PAR, int KS>
__device__ __forceinline__ void ks_steps(const unsigned short* __restrict__ As, const KsTask& T, int c, int wq,
                                         int lane, int fr, int fg, f4 (&acc)[RB][2], u4v (&b0)[3][2],
                                         u4v (&b1)[3][2]) {
  if constexpr (KS < NKS) {
    if constexpr (((KS + PAR) & 1) == 0) ks_step<S, RB, NKS, KS>(As, T, c, wq, lane, fr, fg, acc, b0, b1);
    else ks_step<S, RB, NKS, KS>(As, T, c, wq, lane, fr, fg, acc, b1, b0);
    ks_steps<S, RB, NKS, PAR, KS + 1>(As, T, c, wq, lane, fr, fg, acc, b0, b1);
  }
}

// lane l of each row of 16 takes lane l ^ 8's value (a rotation by 8)
__device__ __forceinline__ f4 ks_swap8(const f4 v) {
  f4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    r[q] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v[q]), 0x128, 0xf, 0xf, false));
  return r;
}

// this wavefront's 16 RB x 32 part of column tile c
template <class S, int RB, int NKS, int PAR>
__device__ __forceinline__ void ks_tile(const unsigned short* __restrict__ As, const KsTask& T, float* y,
                                        const float* __restrict__ bias, float alpha, bool vst, int c, int wq,
                                        int lane, int fr, int fg, u4v (&b0)[3][2], u4v (&b1)[3][2]) {
  const bool has_bias = T.bias_off >= 0;
  // the bias of this lane's 8 columns, loaded before the MFMAs: a load
  // waited for in the stores would wait for the B fragments loaded after it
  f4 bv[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) bv[j] = f4{0.f, 0.f, 0.f, 0.f};
  if (has_bias) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) bv[j][q] = bias[T.bias_off + min(c + 32 * wq + 16 * j + 4 * fg + q, T.ce - 1)];
  }
  f4 acc[RB][2];
  if (T.addend) {
    const bool avec = ((T.n & 3) == 0) && ((T.out_base & 3) == 0) && ((((uintptr_t)T.addend) & 15) == 0);
    const float ia = 1.f / alpha;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = 16 * i + fr, col = c + 32 * wq + 16 * j + 4 * fg;
        acc[i][j] = addend_init(T.addend, T.out_base + (int64_t)r * T.n + col, r < T.rows, col, T.ce, avec, ia);
      }
  } else {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  }
  ks_steps<S, RB, NKS, PAR, 0>(As, T, c, wq, lane, fr, fg, acc, b0, b1);
  // acc[i][j][q] = out[row 16 i + fr][column c + 32 wq + 16 j + 4 fg + q].
  // Lanes fr and fr ^ 8 trade one block, so that a store writes 8 whole rows
  // of the 32 columns (128 contiguous bytes each) instead of 16 half rows:
  // lane fr < 8 keeps j = 0 of row fr and takes j = 0 of row fr + 8; lane
  // fr >= 8 keeps j = 1 of row fr and takes j = 1 of row fr - 8.
  const bool lo = fr < 8;
  const int jl = lo ? 0 : 1;   // this lane's 16-column half, in both stores
  const int col = c + 32 * wq + 16 * jl + 4 * fg;
  // whole 32 columns, 16-byte stores: no test but the row's, one 32-bit lane offset
  const bool whole = vst && c + 32 * wq + 32 <= T.ce;
  const unsigned off = (unsigned)(fr & 7) * (unsigned)T.n + (unsigned)col;
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    f4 v0 = acc[i][0], v1 = acc[i][1];
    if (has_bias) {
      v0 += bv[0];
      v1 += bv[1];
    }
    v0 *= alpha;
    v1 *= alpha;
    const f4 got = ks_swap8(lo ? v1 : v0);
    const f4 s0 = lo ? v0 : got, s1 = lo ? got : v1;   // rows 16 i + (fr & 7), + 8
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = 16 * i + 8 * h + (fr & 7);
      const f4 v = h ? s1 : s0;
      float* yr = y + T.out_base + (int64_t)(16 * i + 8 * h) * T.n;
      if (whole) {
        if (r < T.rows) *(f4*)(yr + off) = v;
      } else if (r < T.rows && col < T.ce) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (col + q < T.ce) yr[off + q] = v[q];
      }
    }
  }
}

template <class S, int RB, int NKS>
__device__ __forceinline__ void ks_columns(const unsigned short* __restrict__ As, const KsTask& T,
                                           float* y, const float* __restrict__ bias, float alpha, int grp,
                                           int wq, int lane, int fr, int fg) {
  int c0 = T.cb + 128 * grp;
  if (c0 >= T.ce) return;
  // 16-byte stores when every 4-column group of every row is 16-byte aligned
  const bool vst = ((T.n & 3) == 0) && ((T.out_base & 3) == 0) && ((T.cb & 3) == 0) && ((((uintptr_t)y) & 15) == 0);
  u4v b0[3][2], b1[3][2];
  if (NKS > 0) ks_load_b(T, c0, 0, wq, lane, b0);
  for (; c0 < T.ce; c0 += 2 * S::CSTEP) {
    ks_tile<S, RB, NKS, 0>(As, T, y, bias, alpha, vst, c0, wq, lane, fr, fg, b0, b1);
    if (c0 + S::CSTEP < T.ce)
      ks_tile<S, RB, NKS, NKS & 1>(As, T, y, bias, alpha, vst, c0 + S::CSTEP, wq, lane, fr, fg, b0, b1);
  }
}

template <class S>
__global__ __launch_bounds__(S::THREADS, S::WAVES) void k_seg_linear_ks(const float* __restrict__ x, float* y,
                                                       const float* addend,
                                                       const unsigned short* __restrict__ wfrag,
                                                       const float* __restrict__ bias,
                                                       const int64_t* __restrict__ tasks, float alpha, int n_tasks,
                                                       int per) {
  constexpr int R = S::R, KM = S::KM;
  __shared__ __attribute__((aligned(16))) unsigned short As[3 * S::PL];
  const int task = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (task >= n_tasks) return;
  const int64_t* td = tasks + 10 * (int64_t)task;
  KsTask T;
  T.out_base = td[0];
  T.rows = (int)td[1];
  if (T.rows <= 0) return;   // a padding entry of the table
  T.n = (int)td[2];
  T.cb = (int)td[3];
  T.ce = (int)td[4];
  T.bias_off = td[5];
  const int64_t x_base = td[6];
  const int k = (int)td[7];
  T.wf = wfrag + td[8];
  T.addend = addend;
  T.nks = (k + 31) >> 5;
  T.nb16 = (T.n + 15) >> 4;
  const int t = (int)threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int grp = wv >> 2, wq = wv & 3;
  const int fr = lane & 15, fg = lane >> 4;
  if (k < 0 || k > KM || T.rows > R) {
    // a k or a height beyond this instantiation's: NaN outputs instead of a
    // product of a truncated A tile (the host table builder never makes such tasks)
    for (int u = t; u < T.rows * (T.ce - T.cb); u += S::THREADS) {
      const int r = u / (T.ce - T.cb), c = T.cb + (u - r * (T.ce - T.cb));
      y[T.out_base + (int64_t)r * T.n + c] = __builtin_nanf("");
    }
    return;
  }

  // A: rows x k of x (row stride k) -> planes, zeros past rows and past k
  // (up to the next multiple of 32)
  {
    const float* __restrict__ xa = x + x_base;
    const bool xvec = ((((uintptr_t)xa) & 15) == 0) && ((k & 3) == 0);
    const int kq = T.nks * 4;   // 8-k units per row
    constexpr int NU = R * KM / 8 / S::THREADS;   // units per thread at most
    auto put = [&](int r, int kk, const f4& a0, const f4& a1) {
      const float v[8] = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
      bx3_bf8 tt[3];
      bx3_split8(v, tt);
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) *(bx3_bf8*)&As[pl * S::PL + r * S::STR + kk] = tt[pl];
    };
    if (xvec && (k & 7) == 0 && k > 0) {
      // every load in flight before the first split: unconditional, the row
      // clamped to the last one (its outputs are not stored) and the 8-k unit
      // into the row (zeros past k: an infinity there would meet zero weights)
      f4 a[NU][2];
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        const int u = min(t + S::THREADS * i, R * kq - 1), r = u / kq, kk = (u - r * kq) * 8;
        const float* p = xa + (int64_t)min(r, T.rows - 1) * k + min(kk, k - 8);
        a[i][0] = *(const f4*)p;
        a[i][1] = *(const f4*)(p + 4);
      }
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        const int u = t + S::THREADS * i, r = u / kq, kk = (u - r * kq) * 8;
        if (u >= R * kq) continue;
        if (kk >= k) a[i][0] = a[i][1] = f4{0.f, 0.f, 0.f, 0.f};
        put(r, kk, a[i][0], a[i][1]);
      }
    } else {
      for (int u = t; u < R * kq; u += S::THREADS) {
        const int r = u / kq, kk = (u - r * kq) * 8;
        const bool ok = r < T.rows;
        const float* p = xa + (int64_t)r * k + kk;
        put(r, kk, seg_ld4(p, ok && xvec && kk + 4 <= k, ok && kk < k, k - kk),
            seg_ld4(p + 4, ok && xvec && kk + 8 <= k, ok && kk + 4 < k, k - kk - 4));
      }
    }
  }
  __syncthreads();

#define KS_C(n)                                                                                                       \
  do {                                                                                                                \
    if (T.rows > 32) ks_columns<S, S::RB, (n) <= KM / 32 ? (n) : 0>(As, T, y, bias, alpha, grp, wq, lane, fr, fg);     \
    else ks_columns<S, 2, (n) <= KM / 32 ? (n) : 0>(As, T, y, bias, alpha, grp, wq, lane, fr, fg);                     \
  } while (0)
  switch (T.nks) {
    case 1: KS_C(1); break;
    case 2: KS_C(2); break;
    case 3: KS_C(3); break;
    case 4: KS_C(4); break;
    case 5: KS_C(5); break;
    case 6: KS_C(6); break;
    case 7: KS_C(7); break;
    case 8: KS_C(8); break;
    default: ks_columns<S, S::RB, 0>(As, T, y, bias, alpha, grp, wq, lane, fr, fg); break;   // k = 0: bias or zeros
  }
#undef KS_C
}

// Per block (6 x int64): src_off, cols, k, transpose, dst_off, layout; one
// double scale.  B[kk][c] = scale * (transpose ? w[src_off + kk cols + c] :
// w[src_off + c k + kk]), zero past k (and past cols).
//  layout 0: column c, k index kk < k_pad = ceil8(k) of term p at
//            out[p * pstride + dst_off + c k_pad + kk];
//  layout 1: MFMA fragment order for k_seg_linear_ks, one buffer: per
//            16-column block cb and 32-k step s (nks = ceil(k / 32) steps),
//            the three terms as 512-element runs in lane order, element
//            (c, kk) of term p at out[dst_off + ((cb nks + s) 3 + p) 512 +
//            (((kk % 32) / 8) 16 + c % 16) 8 + kk % 8], cb = c / 16, s = kk /
//            32, over ceil16(cols) columns.
// blockIdx.y picks the block, the x dimension strides over its elements.
__global__ __launch_bounds__(256) void k_split_blocks(const float* __restrict__ w, const int64_t* __restrict__ blocks,
                                                      const double* __restrict__ scales,
                                                      unsigned short* __restrict__ out, int64_t pstride) {
  const int64_t* bd = blocks + 6 * (int64_t)blockIdx.y;
  const int64_t src = bd[0], dst = bd[4];
  const int cols = (int)bd[1], k = (int)bd[2];
  const bool tr = bd[3] != 0;
  const bool frag = bd[5] == 1;
  const int kpad = frag ? (k + 31) & ~31 : (k + 7) & ~7;
  const int ccols = frag ? (cols + 15) & ~15 : cols;
  const float sc = (float)scales[blockIdx.y];
  const int64_t total = (int64_t)ccols * kpad;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
    const int c = (int)(e / kpad), kk = (int)(e - (int64_t)c * kpad);
    float v = 0.f;
    if (kk < k && c < cols)
      v = bx3_scale2(bx3_f2{tr ? w[src + (int64_t)kk * cols + c] : w[src + (int64_t)c * k + kk], 0.f}, sc).x;
    unsigned h[3];
    bx3_split2(bx3_f2{v, 0.f}, h);
    if (frag) {
      const int64_t run = ((int64_t)(c >> 4) * (kpad >> 5) + (kk >> 5)) * 3;
      const int64_t lane_el = (int64_t)((((kk & 31) >> 3) << 4) + (c & 15)) * 8 + (kk & 7);
#pragma unroll
      for (int p = 0; p < 3; ++p) out[dst + (run + p) * 512 + lane_el] = (unsigned short)(h[p] & 0xffffu);
    } else {
#pragma unroll
      for (int p = 0; p < 3; ++p) out[p * pstride + dst + e] = (unsigned short)(h[p] & 0xffffu);
    }
  }
}

// Several GEMM operands laid out in one launch, each from up to four scaled
// weight matrices stacked along its columns or its rows.  An operand is 20 x
// int64: kind (0 bf16 in MFMA fragment order, 1 three bf16 terms in fragment
// order, 2 float32 row-major [k, n]), k, n, byte offset in out (16-byte
// aligned), segments, axis (0: stacked along n, 1: along k), trans (B[kk][c] =
// W[c][kk], else W[kk][c]), row stride of every W, then per segment its
// address, its length along the axis and its scale (a double's bits).  A
// thread makes the eight values of one lane's fragment (or one float), so its
// stores are 16 bytes; blockIdx.y picks the operand.  The operands come as a
// kernel argument, 24 a launch: a launch, recorded or not, holds its own, and
// no address is kept in memory between calls.
struct OpDesc {
  int64_t d[20];

  __device__ __forceinline__ float at(int kk, int c) const {
    int a = d[5] == 0 ? c : kk, first = 0;   // the index in its segment
    const float* W = (const float*)d[8];
    float sc = (float)__longlong_as_double(d[10]);
#pragma unroll
    for (int s = 1; s < 4; ++s) {
      first += (int)d[6 + 3 * s];   // the lengths of the segments before s
      if (s < (int)d[4] && (d[5] == 0 ? c : kk) >= first) {
        a = (d[5] == 0 ? c : kk) - first;
        W = (const float*)d[8 + 3 * s];
        sc = (float)__longlong_as_double(d[10 + 3 * s]);
      }
    }
    if (d[5] == 0) c = a;
    else kk = a;
    // trans: W's rows are B's columns
    return bx3_scale2(bx3_f2{W[d[6] ? (int64_t)c * d[7] + kk : (int64_t)kk * d[7] + c], 0.f}, sc).x;
  }
};

constexpr int OPS_LAUNCH = 24;
constexpr float BF16_MAX = 0x1.fep127f;
struct OpTable {   // 3,840 bytes
  OpDesc op[OPS_LAUNCH];
};

__global__ __launch_bounds__(256) void k_layout_operands(const OpTable table, unsigned char* __restrict__ out) {
  const OpDesc& o = table.op[blockIdx.y];   // uniform: in scalar registers
  const int kind = (int)o.d[0], k = (int)o.d[1], n = (int)o.d[2];
  unsigned char* dst = out + o.d[3];
  if (kind == 2) {
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < (int64_t)k * n; e += (int64_t)gridDim.x * 256)
      ((float*)dst)[e] = o.at((int)(e / n), (int)(e % n));
    return;
  }
  const int nks = (k + 31) >> 5, nb = (n + 15) >> 4;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < (int64_t)nks * nb * 64; e += (int64_t)gridDim.x * 256) {
    const int lane = (int)(e & 63);
    const int64_t run = e >> 6;   // column block x k step
    const int s = (int)(run % nks), cb = (int)(run / nks);
    const int c = 16 * cb + (lane & 15), k0 = 32 * s + 8 * (lane >> 4);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = c < n && k0 + j < k ? o.at(k0 + j, c) : 0.f;
    bx3_bf8 h[3];
    bx3_split8(v, h);
    if (kind == 0) {
      *(bx3_bf8*)(dst + 1024 * run + 16 * lane) = h[0];
    } else {
      // a weight that rounds past bf16's largest has that as its first term
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (__builtin_isinf((float)h[0][j]) && __builtin_isfinite(v[j])) {
          h[0][j] = (__bf16)(v[j] < 0.f ? -BF16_MAX : BF16_MAX);
          const float r = v[j] - (float)h[0][j];
          h[1][j] = (__bf16)r;
          h[2][j] = (__bf16)(r - (float)h[1][j]);
        }
      }
#pragma unroll
      for (int p = 0; p < 3; ++p) *(bx3_bf8*)(dst + 1024 * (3 * run + p) + 16 * lane) = h[p];
    }
  }
}

}  // namespace

extern "C" int tace_layout_operands(const int64_t* table, int64_t n_operands, void* out, int64_t out_bytes,
                                    void* stream) {
  if (n_operands < 0 || n_operands > 65535) return tace_fail_msg("tace_layout_operands: 0..65535 operands");
  if (n_operands == 0) return 0;
  if (!table || !out || (((uintptr_t)out) & 15) != 0)
    return tace_fail_msg("tace_layout_operands: null or misaligned pointer");
  for (int64_t i = 0; i < n_operands; ++i) {
    const int64_t* d = table + 20 * i;
    if (d[0] < 0 || d[0] > 2 || d[1] <= 0 || d[2] <= 0 || d[1] > 0xffffff || d[2] > 0xffffff || d[4] < 1 || d[4] > 4 ||
        d[5] < 0 || d[5] > 1 || d[3] < 0 || (d[3] & 15) != 0)
      return tace_fail_msg("tace_layout_operands: bad operand");
    const int64_t frag = 1024 * ((d[1] + 31) / 32) * ((d[2] + 15) / 16);
    if (d[3] + (d[0] == 0 ? frag : d[0] == 1 ? 3 * frag : 4 * d[1] * d[2]) > out_bytes)
      return tace_fail_msg("tace_layout_operands: an operand ends past out");
    int64_t along = 0;
    for (int64_t s = 0; s < d[4]; ++s) {
      if (!d[8 + 3 * s] || d[9 + 3 * s] <= 0) return tace_fail_msg("tace_layout_operands: bad segment");
      along += d[9 + 3 * s];
    }
    if (along != (d[5] == 0 ? d[2] : d[1]))
      return tace_fail_msg("tace_layout_operands: the segments are not the operand's length");
  }
  for (int64_t i = 0; i < n_operands; i += OPS_LAUNCH) {
    OpTable t;
    const int m = (int)(n_operands - i < OPS_LAUNCH ? n_operands - i : OPS_LAUNCH);
    memset(&t, 0, sizeof(t));
    memcpy(&t, table + 20 * i, sizeof(OpDesc) * m);
    hipLaunchKernelGGL(k_layout_operands, dim3(64, (unsigned)m), dim3(256), 0, (hipStream_t)stream, t,
                       (unsigned char*)out);
    if (int rc = tace_check_launch("tace_layout_operands")) return rc;
  }
  return 0;
}

extern "C" int tace_bf16x3_split_blocks(const float* w, const int64_t* blocks, const double* scales,
                                        int64_t n_blocks, uint16_t* planes, int64_t plane_stride, void* stream) {
  if (n_blocks < 0 || n_blocks > 65535) return tace_fail_msg("tace_bf16x3_split_blocks: 0..65535 blocks");
  if (n_blocks == 0) return 0;
  if (!w || !blocks || !scales || !planes) return tace_fail_msg("tace_bf16x3_split_blocks: null pointer");
  if (plane_stride < 0) return tace_fail_msg("tace_bf16x3_split_blocks: bad plane stride");
  hipLaunchKernelGGL(k_split_blocks, dim3(64, (unsigned)n_blocks), dim3(256), 0, (hipStream_t)stream, w, blocks,
                     scales, (unsigned short*)planes, plane_stride);
  return tace_check_launch("tace_bf16x3_split_blocks");
}

extern "C" int tace_seg_linear_presplit(const float* x, float* y, const float* addend, const uint16_t* w_planes,
                                        int64_t plane_stride, const float* bias, const int64_t* tiles,
                                        int64_t n_tiles, const int64_t* contribs, double alpha, void* stream) {
  if (n_tiles < 0 || n_tiles > 0x7ffffff0) return tace_fail_msg("tace_seg_linear_presplit: bad tile count");
  if (n_tiles == 0) return 0;
  if (!x || !y || !w_planes || !tiles || !contribs) return tace_fail_msg("tace_seg_linear_presplit: null pointer");
  if ((((uintptr_t)w_planes) & 15) != 0 || (plane_stride & 7) != 0)
    return tace_fail_msg("tace_seg_linear_presplit: planes must be 16-byte aligned with a stride that is a multiple of 8");
  const int per = (int)((n_tiles + 7) / 8);
  hipLaunchKernelGGL(k_seg_linear_bx3s, dim3((unsigned)(8 * per)), dim3(256), 0, (hipStream_t)stream, x, y,
                     addend, (const unsigned short*)w_planes, plane_stride, bias, tiles, contribs, (float)alpha,
                     (int)n_tiles, per);
  return tace_check_launch("tace_seg_linear_presplit");
}

extern "C" int tace_seg_linear_presplit_frag(const float* x, float* y, const float* addend, const uint16_t* w_frag,
                                             const float* bias,
                                             const int64_t* tiles, int64_t n_tiles, const int64_t* contribs,
                                             int32_t aligned, double alpha, void* stream) {
  if (n_tiles < 0 || n_tiles > 0x7ffffff) return tace_fail_msg("tace_seg_linear_presplit_frag: bad tile count");
  if (n_tiles == 0) return 0;
  if (!x || !y || !w_frag || !tiles || !contribs) return tace_fail_msg("tace_seg_linear_presplit_frag: null pointer");
  if (addend && alpha == 0.0) return tace_fail_msg("tace_seg_linear_presplit_frag: an addend needs alpha != 0");
  if ((((uintptr_t)w_frag) & 15) != 0)
    return tace_fail_msg("tace_seg_linear_presplit_frag: fragment-order weights must be 16-byte aligned");
  const int per = (int)((n_tiles + 7) / 8);
  const dim3 g((unsigned)(16 * per)), b(256);   // two 64-row halves per tile
  if (aligned && (((uintptr_t)x) & 15) == 0)
    hipLaunchKernelGGL((k_seg_linear_bx3f<true, false>), g, b, 0, (hipStream_t)stream, x, y, addend,
                       (const unsigned short*)w_frag,
                       bias, tiles, contribs, (float)alpha, (int)n_tiles, per, 1, nullptr, FtDense{0, 0, 0});
  else
    hipLaunchKernelGGL((k_seg_linear_bx3f<false, false>), g, b, 0, (hipStream_t)stream, x, y, addend,
                       (const unsigned short*)w_frag,
                       bias, tiles, contribs, (float)alpha, (int)n_tiles, per, 1, nullptr, FtDense{0, 0, 0});
  return tace_check_launch("tace_seg_linear_presplit_frag");
}

extern "C" int tace_seg_linear_presplit_frag_split(const float* x, float* y, const float* addend,
                                                   const uint16_t* w_frag, const float* bias, const int64_t* tiles,
                                                   int64_t n_tiles, const int64_t* contribs, int32_t aligned,
                                                   int32_t splits, float* partials, int64_t partial_elems,
                                                   double alpha, void* stream) {
  if (n_tiles < 0 || n_tiles > 0x7ffffff0) return tace_fail_msg("tace_seg_linear_presplit_frag_split: bad tile count");
  if (splits < 2 || splits > 64) return tace_fail_msg("tace_seg_linear_presplit_frag_split: 2..64 splits");
  if (n_tiles * splits > 0x7ffffff || n_tiles > 0x7ffffff)
    return tace_fail_msg("tace_seg_linear_presplit_frag_split: too many work items");
  if (n_tiles == 0) return 0;
  if (!x || !y || !w_frag || !tiles || !contribs || !partials)
    return tace_fail_msg("tace_seg_linear_presplit_frag_split: null pointer");
  if (addend && alpha == 0.0) return tace_fail_msg("tace_seg_linear_presplit_frag_split: an addend needs alpha != 0");
  if ((((uintptr_t)w_frag) & 15) != 0 || (((uintptr_t)partials) & 15) != 0)
    return tace_fail_msg("tace_seg_linear_presplit_frag_split: weights and partials must be 16-byte aligned");
  if (partial_elems < n_tiles * splits * 16384)
    return tace_fail_msg("tace_seg_linear_presplit_frag_split: partials hold fewer than n_tiles * splits * 16384 floats");
  const int64_t items = n_tiles * splits;
  const int per = (int)((items + 7) / 8);
  const dim3 g((unsigned)(16 * per)), b(256);   // two 64-row halves per item
  if (aligned && (((uintptr_t)x) & 15) == 0)
    hipLaunchKernelGGL((k_seg_linear_bx3f<true, true>), g, b, 0, (hipStream_t)stream, x, y, addend,
                       (const unsigned short*)w_frag, bias, tiles, contribs, (float)alpha, (int)n_tiles, per,
                       (int)splits, partials, FtDense{0, 0, 0});
  else
    hipLaunchKernelGGL((k_seg_linear_bx3f<false, true>), g, b, 0, (hipStream_t)stream, x, y, addend,
                       (const unsigned short*)w_frag, bias, tiles, contribs, (float)alpha, (int)n_tiles, per,
                       (int)splits, partials, FtDense{0, 0, 0});
  if (int rc = tace_check_launch("tace_seg_linear_presplit_frag_split")) return rc;
  hipLaunchKernelGGL(k_seg_split_sum, dim3((unsigned)(16 * n_tiles)), dim3(256), 0, (hipStream_t)stream, y, addend, bias,
                     tiles, (const float*)partials, (int)splits, (float)alpha);
  return tace_check_launch("tace_seg_linear_presplit_frag_split");
}

extern "C" int tace_gemm_bx3(const float* x, const uint16_t* w_frag, const float* bias, float* y, int64_t m, int32_t n,
                             int32_t k, void* stream) {
  if (m < 0 || n <= 0 || k <= 0) return tace_fail_msg("tace_gemm_bx3: bad sizes");
  const int64_t items = ((m + 127) / 128) * ((n + 127) / 128);
  if (items > 0x7ffffff) return tace_fail_msg("tace_gemm_bx3: too many tiles");
  if (m == 0) return 0;
  if (!x || !w_frag || !y) return tace_fail_msg("tace_gemm_bx3: null pointer");
  if ((((uintptr_t)w_frag) & 15) != 0) return tace_fail_msg("tace_gemm_bx3: the weights must be 16-byte aligned");
  const int per = (int)((items + 7) / 8);
  const dim3 g((unsigned)(16 * per)), b(256);   // two 64-row halves per tile
  const unsigned short* wf = (const unsigned short*)w_frag;
  const FtDense d{m, n, k};
  if ((k & 3) == 0 && (((uintptr_t)x) & 15) == 0)
    hipLaunchKernelGGL((k_seg_linear_bx3f<true, false>), g, b, 0, (hipStream_t)stream, x, y, nullptr, wf, bias, nullptr,
                       nullptr, 1.f, (int)items, per, 1, nullptr, d);
  else
    hipLaunchKernelGGL((k_seg_linear_bx3f<false, false>), g, b, 0, (hipStream_t)stream, x, y, nullptr, wf, bias, nullptr,
                       nullptr, 1.f, (int)items, per, 1, nullptr, d);
  return tace_check_launch("tace_gemm_bx3");
}

extern "C" int32_t tace_seg_linear_ks_rows(int32_t k) { return k >= 0 && k <= 256 ? 64 : 0; }

template <class S>
static void launch_ks(const float* x, float* y, const float* addend, const uint16_t* w_frag, const float* bias,
                      const int64_t* tasks, double alpha, int64_t n_tasks, int per, void* stream) {
  hipLaunchKernelGGL(k_seg_linear_ks<S>, dim3((unsigned)(8 * per)), dim3(S::THREADS), 0, (hipStream_t)stream, x, y,
                     addend, (const unsigned short*)w_frag, bias, tasks, (float)alpha, (int)n_tasks, per);
}

extern "C" int tace_seg_linear_presplit_ks(const float* x, float* y, const float* addend, const uint16_t* w_frag,
                                           const float* bias,
                                           const int64_t* tasks, int64_t n_tasks, int32_t k_max, double alpha,
                                           void* stream) {
  if (k_max != 128 && k_max != 256) return tace_fail_msg("tace_seg_linear_presplit_ks: k_max 128 or 256");
  if (n_tasks < 0 || n_tasks > 0x7ffffff0) return tace_fail_msg("tace_seg_linear_presplit_ks: bad task count");
  if (n_tasks == 0) return 0;
  if (!x || !y || !w_frag || !tasks) return tace_fail_msg("tace_seg_linear_presplit_ks: null pointer");
  if (addend && alpha == 0.0) return tace_fail_msg("tace_seg_linear_presplit_ks: an addend needs alpha != 0");
  if ((((uintptr_t)w_frag) & 15) != 0)
    return tace_fail_msg("tace_seg_linear_presplit_ks: the fragment-order weights must be 16-byte aligned");
  const int per = (int)((n_tasks + 7) / 8);
  if (k_max == 128) launch_ks<KsShape<64, 128, 1>>(x, y, addend, w_frag, bias, tasks, alpha, n_tasks, per, stream);
  else launch_ks<KsShape<64, 256, 2>>(x, y, addend, w_frag, bias, tasks, alpha, n_tasks, per, stream);
  return tace_check_launch("tace_seg_linear_presplit_ks");
}

extern "C" int tace_seg_linear(int dtype, int32_t tile_rows, int32_t tile_cols, const void* x, void* y,
                               const void* addend, const void* w, const void* bias, const int64_t* tiles, int64_t n_tiles,
                               const int64_t* contribs, const double* scales, double alpha, void* stream) {
  if (n_tiles < 0 || n_tiles > 0x7ffffff0) return tace_fail_msg("tace_seg_linear: bad tile count");
  const int tr = tile_rows, tc = tile_cols;
  const bool mfma = dtype == TACE_F32 && tr == 128 && tc == 128;
  if (!(mfma || ((dtype == TACE_F32 || dtype == TACE_F64) && tr == 64 && tc == 64)))
    return tace_fail_msg("tace_seg_linear: tiles must be 128x128 (float32) or 64x64");
  if (n_tiles == 0) return 0;
  if (!x || !y || !w || !tiles || !contribs || !scales) return tace_fail_msg("tace_seg_linear: null pointer");
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)n_tiles), block(256);
  if (mfma) {
    const int per = (int)((n_tiles + 7) / 8);
    const dim3 g8((unsigned)(8 * per));
    hipLaunchKernelGGL(k_seg_linear_bf16x3, g8, block, 0, s, (const float*)x, (float*)y, (const float*)addend,
                       (const float*)w,
                       (const float*)bias, tiles, contribs, scales, (float)alpha, (int)n_tiles, per);
  } else if (dtype == TACE_F32)
    hipLaunchKernelGGL(k_seg_linear<float>, grid, block, 0, s, (const float*)x, (float*)y, (const float*)addend,
                       (const float*)w,
                       (const float*)bias, tiles, contribs, scales, (float)alpha);
  else if (dtype == TACE_F64)
    hipLaunchKernelGGL(k_seg_linear<double>, grid, block, 0, s, (const double*)x, (double*)y,
                       (const double*)addend, (const double*)w,
                       (const double*)bias, tiles, contribs, scales, alpha);
  else
    return tace_fail_msg("tace_seg_linear: dtype must be TACE_F32 or TACE_F64");
  return tace_check_launch("tace_seg_linear");
}
