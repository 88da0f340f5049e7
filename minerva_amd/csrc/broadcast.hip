// Broadcast ("norm") arithmetic on a column-major {m,n} matrix: the matrix is
// combined with a vector that is replicated along one dimension (reference
// minerva/op/impl/basic.cpp:319-367; CUDA kernels cuda_kernel.h:107-130).
// HBM stream, 8 bytes per element (+ the vector, which stays in cache).
//   col variant: vec has n entries, one per column  -> res[r + c*m] = M[r + c*m] (op) vec[c]
//   row variant: vec has m entries, one per row     -> res[r + c*m] = M[r + c*m] (op) vec[r]
// Work is laid out as (column, 1 KiB row segment) tiles so every wavefront access is
// contiguous and no thread divides by m.
#include "mnv_common.h"

namespace {

struct OpAdd { __device__ float operator()(float a, float b) const { return a + b; } };
struct OpSub { __device__ float operator()(float a, float b) const { return a - b; } };
struct OpMul { __device__ float operator()(float a, float b) const { return a * b; } };
struct OpDiv { __device__ float operator()(float a, float b) const { return a / b; } };

#define MNV_BC_THREADS 256
#define MNV_BC_COLS 4  // columns per workgroup iteration: 4 independent 16-byte loads in flight

// ROWVEC = true: vector indexed by row (shape {m,1}); false: by column ({1,n}).
// W = 4: rows per thread.  VEC4: every column starts on the 16-byte grid; otherwise the same 16-byte
// accesses at the addresses the columns have (4 bytes per access before: 8191 x 8193 116 -> 107
// us), and the thread whose rows a column's end cuts loads the column's last four values and stores
// those of them that are its own.
// W = 1: one row per thread, for columns of a few rows.
template <class Op, bool ROWVEC, int W, bool VEC4, bool NT>
__global__ __launch_bounds__(MNV_BC_THREADS) void mnv_norm_kernel(
    const float* __restrict__ mat, const float* __restrict__ vec, float* __restrict__ res, int m,
    int n, Op op) {
  const int r0 = (blockIdx.x * blockDim.x + threadIdx.x) * W;
  if (r0 >= m) return;
  const int skip = W == 4 && !VEC4 && r0 + 3 >= m ? r0 + 4 - m : 0, rb = r0 - skip;  // m >= 4 here
  float rv[W];
  if (ROWVEC) {
#pragma unroll
    for (int q = 0; q < W; ++q) rv[q] = vec[rb + q];
  }
  for (int c0 = blockIdx.y * MNV_BC_COLS; c0 < n; c0 += gridDim.y * MNV_BC_COLS) {
    if constexpr (W == 4) {
      mnv_f4 v[MNV_BC_COLS];
#pragma unroll
      for (int u = 0; u < MNV_BC_COLS; ++u)
        if (c0 + u < n)
          v[u] = VEC4 ? mnv_ldx4<NT>(reinterpret_cast<const mnv_f4*>(mat + (size_t)(c0 + u) * m + rb))
                      : mnv_ldx4u<NT>(mat + (size_t)(c0 + u) * m + rb);
#pragma unroll
      for (int u = 0; u < MNV_BC_COLS; ++u)
        if (c0 + u < n) {
          float cv = ROWVEC ? 0.f : vec[c0 + u];
          mnv_f4 o;
          o.x = op(v[u].x, ROWVEC ? rv[0] : cv);
          o.y = op(v[u].y, ROWVEC ? rv[1 % W] : cv);
          o.z = op(v[u].z, ROWVEC ? rv[2 % W] : cv);
          o.w = op(v[u].w, ROWVEC ? rv[3 % W] : cv);
          float* at = res + (size_t)(c0 + u) * m + rb;
          if (!VEC4 && skip) {
            if (skip < 2) at[1] = o.y;
            if (skip < 3) at[2] = o.z;
            at[3] = o.w;
          } else if (!VEC4) {
            *reinterpret_cast<mnv_f4u*>(at) = o;
          } else if (NT) {
            __builtin_nontemporal_store(o, reinterpret_cast<mnv_f4*>(at));
          } else {
            *reinterpret_cast<mnv_f4*>(at) = o;
          }
        }
    } else {
#pragma unroll
      for (int u = 0; u < MNV_BC_COLS; ++u)
        if (c0 + u < n) {
          const size_t i = (size_t)(c0 + u) * m + r0;
          res[i] = op(mat[i], ROWVEC ? rv[0] : vec[c0 + u]);
        }
    }
  }
}

template <class Op, bool ROWVEC>
int launch_norm(const float* mat, const float* vec, float* res, int m, int n, mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!mat || !vec || !res || m < 0 || n < 0) return MNV_ERR_INVALID;
  const bool vec4 = (m % 4 == 0) && mnv_aligned16(mat) && mnv_aligned16(res);
  // One row per thread below 16 rows off the 16-byte grid (with four: 15 x 1333333 111 us, one 103, and
  // 60 in workgroups of one wavefront; 33 x 606060 44.6 against 52.7).  The workgroups of a column share
  // its rows evenly: a last one with a single row cost a fifth (1025 x 19512 32.6 -> 27.7 us).
  const bool narrow = !vec4 && m < 16;
  const int rows = narrow ? 1 : 4;
  const unsigned vecs = (unsigned)mnv_ceil_div((size_t)m, rows);
  const unsigned gx = (unsigned)mnv_ceil_div(vecs, MNV_BC_THREADS);
  const unsigned threads = (unsigned)mnv_ceil_div(mnv_ceil_div(vecs, gx), MNV_WAVE) * MNV_WAVE;
  // enough column groups to give ~8192 workgroups in total, at most one per column group
  unsigned want = 8192u / gx;
  unsigned gy = (unsigned)mnv_ceil_div((size_t)n, MNV_BC_COLS);
  if (gy > want) gy = want ? want : 1u;
  if (gy > 65535u) gy = 65535u;
  dim3 grid(gx, gy);
  // past the 256 MB last-level cache the matrix streams with non-temporal accesses
  const bool nt = (size_t)m * n * 8 >= ((size_t)512 << 20);
#define MNV_BC_LAUNCH(W, VEC4, NT)                                                              \
  hipLaunchKernelGGL((mnv_norm_kernel<Op, ROWVEC, W, VEC4, NT>), grid, dim3(threads), 0, \
                     mnv_stream(stream), mat, vec, res, m, n, Op())
  if (narrow) MNV_BC_LAUNCH(1, false, false);
  else if (vec4) { if (nt) MNV_BC_LAUNCH(4, true, true); else MNV_BC_LAUNCH(4, true, false); }
  else { if (nt) MNV_BC_LAUNCH(4, false, true); else MNV_BC_LAUNCH(4, false, false); }
#undef MNV_BC_LAUNCH
  return MNV_LAUNCH_STATUS();
}

}  // namespace

extern "C" {
#define MNV_NORM_ENTRY(name, OP, ROWVEC)                                                   \
  int name(const float* matrix, const float* vec, float* res, int m, int n, mnv_stream_t s) { \
    return launch_norm<OP, ROWVEC>(matrix, vec, res, m, n, s);                             \
  }
MNV_NORM_ENTRY(mnv_norm_add_col, OpAdd, false)
MNV_NORM_ENTRY(mnv_norm_sub_col, OpSub, false)
MNV_NORM_ENTRY(mnv_norm_mul_col, OpMul, false)
MNV_NORM_ENTRY(mnv_norm_div_col, OpDiv, false)
MNV_NORM_ENTRY(mnv_norm_add_row, OpAdd, true)
MNV_NORM_ENTRY(mnv_norm_sub_row, OpSub, true)
MNV_NORM_ENTRY(mnv_norm_mul_row, OpMul, true)
MNV_NORM_ENTRY(mnv_norm_div_row, OpDiv, true)
}  // extern "C"
