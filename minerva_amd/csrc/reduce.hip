// Reductions of a column-major {m,n} matrix: sum / max along either dimension,
// arg-max along either dimension, and the convolution bias gradient.
// Roofline: HBM bandwidth, 4 algorithmic bytes per input element.
//
// Reference semantics (minerva/op/impl/basic.cpp:189-217, 369-398): a left fold in
// ascending index order that starts from the first element; max / arg-max use a
// strict '<', so the first occurrence of the maximum wins and a NaN is never
// selected unless it is the first element.  Max and arg-max reproduce that
// exactly under any parallel order by reducing (value, index) pairs: the larger
// value wins, equal values keep the lower index (so the bits of a +0 / -0 tie are
// the reference's), NaNs are skipped, and a NaN in position 0 is restored at the
// end.  Sums are tree-ordered (fp32), which differs from the sequential fold only
// in rounding.
#include <math.h>

#include "mnv_common.h"

namespace {

#define MNV_NONE 0x7fffffff

struct SumAcc {
  static constexpr int ROW_UNROLL = 2;  // columns in flight per thread in the row reducer
  static constexpr int ROW_FEW = 32, ROW_FEW_ODD = 48;  // columns, see launch_reduce_row
  static constexpr bool SKIP_IDLE = false;  // merges of idle lanes cost less than the branches around them
  float s;
  __device__ void init() { s = 0.f; }
  __device__ void push(float v, int) { s += v; }
  __device__ void merge(const SumAcc& o) { s += o.s; }
  __device__ SumAcc shfl_down(int off) const {
    SumAcc r;
    r.s = __shfl_down(s, off, MNV_WAVE);
    return r;
  }
  // first = element 0 of the reduced line (only the pair reducers need it)
  __device__ float result_value(float) const { return s; }
};

struct ArgAcc {
  static constexpr int ROW_UNROLL = 4;
  static constexpr int ROW_FEW = 128, ROW_FEW_ODD = 256;
  static constexpr bool SKIP_IDLE = true;  // 1000000 columns of 1: 136 -> 97 us
  float v;
  int idx;
  __device__ void init() {
    v = -INFINITY;
    idx = MNV_NONE;
  }
  // Elements reach one accumulator in ascending index order.  Selections, no branches: where few
  // lanes have rows, all of them skipping the update is common, and each jump over it stalled the
  // wavefront (36 x 4097 37 us, 32 x 4097 14).
  __device__ void push(float x, int i) {
    const bool take = ((idx == MNV_NONE) & (x == x)) | (x > v);  // v is -inf before the first one
    v = take ? x : v;
    idx = take ? i : idx;
  }
  __device__ void merge(const ArgAcc& o) {
    const bool take = (o.idx != MNV_NONE) & ((idx == MNV_NONE) | (o.v > v) | ((o.v == v) & (o.idx < idx)));
    v = take ? o.v : v;
    idx = take ? o.idx : idx;
  }
  __device__ ArgAcc shfl_down(int off) const {
    ArgAcc r;
    r.v = __shfl_down(v, off, MNV_WAVE);
    r.idx = __shfl_down(idx, off, MNV_WAVE);
    return r;
  }
  __device__ float result_value(float first) const { return (first != first) ? first : v; }
  __device__ float result_index(float first) const {
    return (first != first || idx == MNV_NONE) ? 0.f : (float)idx;
  }
};

// What a reducer writes.
struct EmitValue {
  template <class Acc>
  __device__ static float get(const Acc& a, float first) { return a.result_value(first); }
};
struct EmitIndex {
  __device__ static float get(const ArgAcc& a, float first) { return a.result_index(first); }
};

// ---------------------------------------------------------------------------
// Along dimension 0: each of the n columns is m contiguous floats.
// GROUP threads (one wavefront, or the whole 256-thread workgroup) share a column.
// LOAD: 16-byte loads of columns on the 16-byte grid, the same at whatever address a column has
// (4 bytes at a time, one load in flight before: sums of 8191 x 8193 53 -> 38 us), or one value
// per lane, for columns that are short of a vector per lane anyway.
// ---------------------------------------------------------------------------
#define MNV_RC_THREADS 256
enum RcLoad { RC_SINGLE, RC_ODD, RC_VEC4 };

template <class Acc, class Emit, int GROUP, RcLoad LOAD, bool NT>
__global__ __launch_bounds__(MNV_RC_THREADS) void mnv_reduce_col_kernel(
    const float* __restrict__ in, float* __restrict__ out, int m, int n) {
  constexpr int COLS = MNV_RC_THREADS / GROUP;
  __shared__ Acc part[MNV_RC_THREADS / MNV_WAVE];
  const int g = threadIdx.x / GROUP;
  const int t = threadIdx.x % GROUP;
  const int lanes = LOAD == RC_SINGLE ? m : (m + 3) >> 2;  // lanes from here on have nothing to merge
  for (int c = blockIdx.x * COLS + g; c < n; c += gridDim.x * COLS) {
    const float* col = in + (size_t)c * m;
    Acc acc;
    acc.init();
    if (LOAD == RC_SINGLE) {
      for (int i = t; i < m; i += GROUP) acc.push(col[i], i);
    } else {
      auto ld = [&](int i) {
        return LOAD == RC_VEC4 ? mnv_ldx4<NT>(reinterpret_cast<const mnv_f4*>(col) + i) : mnv_ldx4u<NT>(col + 4 * (size_t)i);
      };
      auto push = [&](const mnv_f4& v, int i) {
        acc.push(v.x, 4 * i); acc.push(v.y, 4 * i + 1); acc.push(v.z, 4 * i + 2); acc.push(v.w, 4 * i + 3);
      };
      const int m4 = m >> 2;
      int i = t;
      // two independent 16-byte loads in flight per thread
      for (; i + GROUP < m4; i += 2 * GROUP) {
        const mnv_f4 a = ld(i), b = ld(i + GROUP);
        push(a, i);
        push(b, i + GROUP);
      }
      if (i < m4) push(ld(i), i);
      if (LOAD == RC_ODD && 4 * m4 + t < m) acc.push(col[4 * m4 + t], 4 * m4 + t);
    }
#pragma unroll
    for (int off = MNV_WAVE / 2; off > 0; off >>= 1)
      if (!Acc::SKIP_IDLE || off < lanes) acc.merge(acc.shfl_down(off));
    if (GROUP > MNV_WAVE) {
      const int w = threadIdx.x / MNV_WAVE;
      if ((threadIdx.x % MNV_WAVE) == 0) part[w] = acc;
      __syncthreads();
      if (threadIdx.x == 0) {
        for (int q = 1; q < MNV_RC_THREADS / MNV_WAVE; ++q) acc.merge(part[q]);
        out[c] = Emit::get(acc, col[0]);
      }
      __syncthreads();
    } else if (t == 0) {
      out[c] = Emit::get(acc, col[0]);
    }
  }
}

template <class Acc, class Emit>
int launch_reduce_col(const float* in, float* out, int m, int n, mnv_stream_t stream) {
  if (n == 0) return MNV_OK;
  if (!in || !out || m <= 0 || n < 0) return MNV_ERR_INVALID;
  hipStream_t s = mnv_stream(stream);
  const bool vec4 = (m % 4 == 0) && mnv_aligned16(in);
  const bool big = (size_t)m * n * sizeof(float) >= MNV_PAST_CACHE_BYTES;
#define MNV_RC_LAUNCH(GROUP, LOAD, NT, GRID)                                                           \
  hipLaunchKernelGGL((mnv_reduce_col_kernel<Acc, Emit, GROUP, LOAD, NT>), dim3(GRID), dim3(MNV_RC_THREADS), \
                     0, s, in, out, m, n)
  if (m > 2048) {
    const unsigned grid = (unsigned)(n < 65536 ? n : 65536);
    if (vec4) { if (big) MNV_RC_LAUNCH(MNV_RC_THREADS, RC_VEC4, true, grid); else MNV_RC_LAUNCH(MNV_RC_THREADS, RC_VEC4, false, grid); }
    else { if (big) MNV_RC_LAUNCH(MNV_RC_THREADS, RC_ODD, true, grid); else MNV_RC_LAUNCH(MNV_RC_THREADS, RC_ODD, false, grid); }
  } else {
    const size_t cols = MNV_RC_THREADS / MNV_WAVE, want = mnv_ceil_div((size_t)n, cols);
    const unsigned grid = (unsigned)(want < 65536 ? want : 65536);
    // off the 16-byte grid one value per lane below 96 (vectors -> values, sums of 100000 columns: of 63
    // 15.6 -> 12.4 us, 79 16.1 -> 15.7, 95 16.5 -> 16.7, 129 17.6 -> 20.3)
    if (vec4) { if (big) MNV_RC_LAUNCH(MNV_WAVE, RC_VEC4, true, grid); else MNV_RC_LAUNCH(MNV_WAVE, RC_VEC4, false, grid); }
    else if (m < 96) MNV_RC_LAUNCH(MNV_WAVE, RC_SINGLE, false, grid);
    else { if (big) MNV_RC_LAUNCH(MNV_WAVE, RC_ODD, true, grid); else MNV_RC_LAUNCH(MNV_WAVE, RC_ODD, false, grid); }
  }
#undef MNV_RC_LAUNCH
  return MNV_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------
// Along dimension 1: out[r] = reduce_c in[r + c*m] (stride m between elements).
// A workgroup owns RL*W consecutive rows (128 contiguous bytes per column) and
// splits the columns over CG thread groups; partial results meet in LDS.
// W = 4 rows per thread; 1 for few columns and for matrices of less than four rows.
// VEC4: m and the matrix on the 16-byte grid; otherwise the same loads at the addresses the
// columns have, and the thread whose rows the matrix ends in reduces its last four rows and keeps
// its own.  (One row per thread, 4 bytes per load, one load in flight: sums of 8191 x 8193
// 140 us, 65 x 4097 27.4; vectors with the last rows element by element 120 and 8.3; now 75 and
// 7.4.  At 8192 x 8192 44: the 128-byte run of an unaligned column lies in two lines, both fetched
// whole.)
// ---------------------------------------------------------------------------
template <class Acc, class Emit, int RL, int CG, int W, bool VEC4, bool NT>
__global__ __launch_bounds__(RL* CG) void mnv_reduce_row_kernel(const float* __restrict__ in,
                                                                float* __restrict__ out, int m,
                                                                int n) {
  constexpr int ROWS = RL * W;
  __shared__ Acc part[CG][ROWS + 1];
  const int rl = threadIdx.x % RL;
  const int cg = threadIdx.x / RL;
  const int r0 = blockIdx.x * ROWS + rl * W;
  const int skip = W == 4 && !VEC4 && r0 + 3 >= m ? r0 + 4 - m : 0;  // rows that are another thread's
  Acc acc[W];
#pragma unroll
  for (int q = 0; q < W; ++q) acc[q].init();
  if (r0 < m) {
    const float* first = in + (r0 - skip);
    if constexpr (W == 4) {
      auto ld = [&](int c) {
        const float* at = first + (size_t)c * m;
        return VEC4 ? mnv_ldx4<NT>(reinterpret_cast<const mnv_f4*>(at)) : mnv_ldx4u<NT>(at);
      };
      // several columns in flight per thread: with one workgroup per 32 rows there are few
      // wavefronts per SIMD, and the loads of a thread are what keeps HBM busy (measured:
      // four for the (value, index) pairs, 4.9 -> 6.0 TB/s; two for sums, where four lose 7%)
      constexpr int U = Acc::ROW_UNROLL;
      int c = cg;
      for (; c + (U - 1) * CG < n; c += U * CG) {
        mnv_f4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          v[u] = ld(c + u * CG);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          acc[0].push(v[u].x, c + u * CG); acc[1].push(v[u].y, c + u * CG);
          acc[2].push(v[u].z, c + u * CG); acc[3].push(v[u].w, c + u * CG);
        }
      }
      for (; c < n; c += CG) {
        mnv_f4 a = ld(c);
        acc[0].push(a.x, c); acc[1].push(a.y, c); acc[2].push(a.z, c); acc[3].push(a.w, c);
      }
    } else {
      for (int c = cg; c < n; c += CG) acc[0].push(first[(size_t)c * m], c);
    }
  }
#pragma unroll
  for (int q = 0; q < W; ++q)
    if (q >= skip) part[cg][rl * W + q - skip] = acc[q];
  __syncthreads();
  for (int sft = CG / 2; sft > 0; sft >>= 1) {
    if (cg < sft) {
#pragma unroll
      for (int q = 0; q < W; ++q) {
        Acc a = part[cg][rl * W + q];
        a.merge(part[cg + sft][rl * W + q]);
        part[cg][rl * W + q] = a;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x < ROWS) {
    int r = blockIdx.x * ROWS + threadIdx.x;
    if (r < m) out[r] = Emit::get(part[0][threadIdx.x], in[r]);
  }
}

template <class Acc, class Emit>
int launch_reduce_row(const float* in, float* out, int m, int n, mnv_stream_t stream) {
  if (m == 0) return MNV_OK;
  if (!in || !out || m < 0 || n <= 0) return MNV_ERR_INVALID;
  hipStream_t s = mnv_stream(stream);
  const bool vec4 = (m % 4 == 0) && mnv_aligned16(in);
  const bool big = (size_t)m * n * sizeof(float) >= MNV_PAST_CACHE_BYTES;
#define MNV_RR_LAUNCH(RL, CG, W, VEC4, NT)                                                            \
  hipLaunchKernelGGL((mnv_reduce_row_kernel<Acc, Emit, RL, CG, W, VEC4, NT>),                          \
                     dim3((unsigned)mnv_ceil_div((size_t)m, RL * W)), dim3(RL * CG), 0, s, in, out, m, n)
  // One row per thread and fewer column groups for few columns, where the groups' sums meeting in LDS
  // are most of the work (four rows and 64 groups -> one and 16, us: sums of 100003 x 9 5.7 -> 3.8,
  // 100000 x 32 5.6 -> 4.4, 100003 x 33 6.6 -> 6.2, 727272 x 33 33.7 -> 37.4, 100003 x 63 9.0 -> 10.3;
  // maxima of 255 x 9 4.0 -> 3.4, 100003 x 17 11.7 -> 5.8, 100000 x 128 17.7 -> 15.6, 15000 x 200 5.9 ->
  // 6.4, 100003 x 129 23.5 -> 20.4, 2049 x 257 4.0 -> 5.0; four groups up to four columns: maxima of
  // 3000001 x 1 91.6 -> 17.3).
  if (n <= 4) MNV_RR_LAUNCH(64, 4, 1, false, false);
  else if (n < (vec4 ? Acc::ROW_FEW : Acc::ROW_FEW_ODD)) MNV_RR_LAUNCH(32, 16, 1, false, false);
  else if (vec4) { if (big) MNV_RR_LAUNCH(8, 64, 4, true, true); else MNV_RR_LAUNCH(8, 64, 4, true, false); }
  else if (m < 4) MNV_RR_LAUNCH(4, 128, 1, false, false);
  else if (big) MNV_RR_LAUNCH(8, 64, 4, false, true);
  else MNV_RR_LAUNCH(8, 64, 4, false, false);
#undef MNV_RR_LAUNCH
  return MNV_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------
// Convolution bias gradient: db[k] = sum over images and positions of dY[n,k,:,:]
// (reference cuda_perform.cu:320-337).  A channel's data is N runs of hw contiguous
// floats, one per image.  Workgroup (k, g) sums channel k over image group g: its four
// wavefronts take the group's images round-robin and read each run with 16-byte loads
// from its first aligned address (at most three single floats on either side).  With
// several groups per channel the group sums go to a scratch area and a second, tiny
// kernel adds them in a fixed order, so the result does not depend on scheduling.
// ---------------------------------------------------------------------------
#define MNV_BIAS_THREADS 256

template <bool NT>
__global__ __launch_bounds__(MNV_BIAS_THREADS) void mnv_conv_bwd_bias_kernel(
    const float* __restrict__ top_diff, float* __restrict__ out, int N, int K, int hw,
    int images_per_group) {
  constexpr int NW = MNV_BIAS_THREADS / MNV_WAVE;
  __shared__ float part[NW];
  const int k = blockIdx.x, g = blockIdx.y;
  const int wave = threadIdx.x / MNV_WAVE, lane = threadIdx.x % MNV_WAVE;
  const int img_end = min(N, (g + 1) * images_per_group);
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  for (int img = g * images_per_group + wave; img < img_end; img += NW) {
    const float* p = top_diff + ((size_t)img * K + k) * hw;
    int head = (int)((4 - ((reinterpret_cast<uintptr_t>(p) >> 2) & 3)) & 3);
    if (head > hw) head = hw;
    const int n4 = (hw - head) >> 2, tail = (hw - head) & 3;
    const mnv_f4* p4 = reinterpret_cast<const mnv_f4*>(p + head);
    float edge0 = 0.f, edge1 = 0.f;  // used after the vectors so that they do not wait for these
    if (lane < head) edge0 = p[lane];
    if (lane < tail) edge1 = p[head + 4 * n4 + lane];
    // Four loads in flight per lane in every iteration, the last one included: a vector
    // past the end of the run is read from the run's last vector instead (a cache hit) and
    // counted as 0, so there is no one-load-at-a-time remainder loop (a run of 55 x 55
    // floats would spend four of its six trips to memory in it).
    if (n4 > 0) {
      const int last = n4 - 1;
      for (int i = lane; i < n4; i += 4 * MNV_WAVE) {
        const int i1 = i + MNV_WAVE, i2 = i + 2 * MNV_WAVE, i3 = i + 3 * MNV_WAVE;
        mnv_f4 a = mnv_ldx4<NT>(p4 + i), b = mnv_ldx4<NT>(p4 + min(i1, last)),
               c = mnv_ldx4<NT>(p4 + min(i2, last)), d = mnv_ldx4<NT>(p4 + min(i3, last));
        s0 += (a.x + a.y) + (a.z + a.w);
        s1 += i1 < n4 ? (b.x + b.y) + (b.z + b.w) : 0.f;
        s2 += i2 < n4 ? (c.x + c.y) + (c.z + c.w) : 0.f;
        s3 += i3 < n4 ? (d.x + d.y) + (d.z + d.w) : 0.f;
      }
    }
    s0 += edge0;
    s1 += edge1;
  }
  float s = mnv_wave_sum((s0 + s1) + (s2 + s3));
  if (lane == 0) part[wave] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int q = 0; q < NW; ++q) t += part[q];
    out[(size_t)k * gridDim.y + g] = t;
  }
}

// One wavefront per channel, a group sum per lane and trip: one trip up to 64 groups, 32 at most (2048
// groups, one channel of 8192 images).  (One thread per channel walked them one trip to memory after
// the other: 64 groups, 16 channels of 256 images, 6.4 -> 2.3 us; with its first kernel, 8192 images of
// one 3 x 3 channel 126 -> 10.9.)
__global__ __launch_bounds__(256) void mnv_conv_bwd_bias_finish_kernel(
    const float* __restrict__ partial, float* __restrict__ bias_diff, int K, int groups) {
  const int k = blockIdx.x * (256 / MNV_WAVE) + threadIdx.x / MNV_WAVE, lane = threadIdx.x % MNV_WAVE;
  if (k >= K) return;
  float t = 0.f;
  for (int g = lane; g < groups; g += MNV_WAVE) t += partial[(size_t)k * groups + g];
  t = mnv_wave_sum(t);
  if (lane == 0) bias_diff[k] = t;
}

// The whole channel in one workgroup, and no second launch, where it is short: the images' planes in vectors of four
// laid end to end, four in flight per thread.  A plane's last vector begins four values before its end and counts
// those that the vector before it has as 0.  hw >= 4.  Bound by a launch and a trip to memory, from 8192 vectors on
// by what one CU reads.  Two launches -> this, us: 312 channels of 64 x 32 values 7.0 -> 3.5, 240 of 222 x 52 12.0 -> 3.5, 24 of
// 154 x 423 (16324 vectors) 6.8 -> 5.4, 344 of 118 x 672 (19824) 19.3 -> 17.7; up to four images, one launch before too, the same.
#define MNV_BIAS_SHORT_VECTORS 16384
__global__ __launch_bounds__(1024) void mnv_conv_bwd_bias_short_kernel(const float* __restrict__ top_diff, float* __restrict__ out,
                                                                       int N, int K, int hw, MnvFastDiv d_vectors) {
  __shared__ float part[1024 / MNV_WAVE];
  const int k = blockIdx.x, per = (hw + 3) / 4, total = N * per;
  const float* p = top_diff + (size_t)k * hw;
  const size_t image = (size_t)K * hw;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  for (int u0 = threadIdx.x; u0 < total; u0 += 4 * 1024) {
    mnv_f4 v[4];
    int skip[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool on = u0 + i * 1024 < total;
      const int u = on ? u0 + i * 1024 : total - 1;
      const int img = mnv_fastdiv(u, d_vectors), at = (u - img * per) * 4, from = at + 4 <= hw ? at : hw - 4;
      v[i] = mnv_ldx4u<false>(p + img * image + from);
      skip[i] = on ? at - from : 4;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      s[i] += ((skip[i] > 0 ? 0.f : v[i].x) + (skip[i] > 1 ? 0.f : v[i].y)) + ((skip[i] > 2 ? 0.f : v[i].z) + (skip[i] > 3 ? 0.f : v[i].w));
  }
  const float sum = mnv_wave_sum((s[0] + s[1]) + (s[2] + s[3]));
  if (threadIdx.x % MNV_WAVE == 0) part[threadIdx.x / MNV_WAVE] = sum;
  __syncthreads();
  if (threadIdx.x >= MNV_WAVE) return;
  const float t = mnv_wave_sum(threadIdx.x < 1024 / MNV_WAVE ? part[threadIdx.x] : 0.f);
  if (threadIdx.x == 0) out[k] = t;
}

// Image groups per channel: enough workgroups to fill the chip, at least four images
// per wavefront's worth of work in each.
int bias_groups(int num_images, int channels) {
  int want = (2048 + channels - 1) / channels;
  int max_groups = (num_images + 3) / 4;
  if (want > max_groups) want = max_groups;
  if (want < 1) want = 1;
  int per = (num_images + want - 1) / want;
  return (num_images + per - 1) / per;
}

}  // namespace

extern "C" {

int mnv_reduce_sum_col(const float* in, float* out, int m, int n, mnv_stream_t s) {
  return launch_reduce_col<SumAcc, EmitValue>(in, out, m, n, s);
}
int mnv_reduce_max_col(const float* in, float* out, int m, int n, mnv_stream_t s) {
  return launch_reduce_col<ArgAcc, EmitValue>(in, out, m, n, s);
}
int mnv_reduce_sum_row(const float* in, float* out, int m, int n, mnv_stream_t s) {
  return launch_reduce_row<SumAcc, EmitValue>(in, out, m, n, s);
}
int mnv_reduce_max_row(const float* in, float* out, int m, int n, mnv_stream_t s) {
  return launch_reduce_row<ArgAcc, EmitValue>(in, out, m, n, s);
}
int mnv_maxindex_col(const float* in, float* out, int m, int n, mnv_stream_t s) {
  return launch_reduce_col<ArgAcc, EmitIndex>(in, out, m, n, s);
}
int mnv_maxindex_row(const float* in, float* out, int m, int n, mnv_stream_t s) {
  return launch_reduce_row<ArgAcc, EmitIndex>(in, out, m, n, s);
}

size_t mnv_conv_bwd_bias_workspace_bytes(int num_images, int top_num_channels) {
  if (num_images <= 0 || top_num_channels <= 0) return 0;
  int groups = bias_groups(num_images, top_num_channels);
  return groups > 1 ? (size_t)groups * top_num_channels * sizeof(float) : 0;
}

int mnv_conv_bwd_bias(const float* top_diff, float* bias_diff, int num_images,
                      int top_num_channels, int top_height, int top_width, void* workspace,
                      size_t workspace_bytes, mnv_stream_t stream) {
  if (top_num_channels == 0) return MNV_OK;
  if (!top_diff || !bias_diff || num_images <= 0 || top_num_channels < 0 || top_height <= 0 ||
      top_width <= 0)
    return MNV_ERR_INVALID;
  long long hw = (long long)top_height * top_width;
  if (hw > 0x7fffffffLL || top_num_channels > 0x7fffffff / 2) return MNV_ERR_INVALID;
  int groups = bias_groups(num_images, top_num_channels);
  if (groups > 65535) groups = 65535;
  if (!workspace || workspace_bytes < (size_t)groups * top_num_channels * sizeof(float)) groups = 1;
  int per = (num_images + groups - 1) / groups;
  hipStream_t s = mnv_stream(stream);
  if (hw >= 4 && bias_groups(num_images, top_num_channels) > 1 && num_images * ((hw + 3) / 4) <= MNV_BIAS_SHORT_VECTORS) {
    hipLaunchKernelGGL(mnv_conv_bwd_bias_short_kernel, dim3(top_num_channels), dim3(1024), 0, s, top_diff, bias_diff, num_images,
                       top_num_channels, (int)hw, mnv_fastdiv_make((int)((hw + 3) / 4)));
    return MNV_LAUNCH_STATUS();
  }
  float* out = groups > 1 ? reinterpret_cast<float*>(workspace) : bias_diff;
  if ((size_t)num_images * top_num_channels * hw * sizeof(float) >= MNV_PAST_CACHE_BYTES)
    hipLaunchKernelGGL(mnv_conv_bwd_bias_kernel<true>, dim3(top_num_channels, groups),
                       dim3(MNV_BIAS_THREADS), 0, s, top_diff, out, num_images, top_num_channels,
                       (int)hw, per);
  else
    hipLaunchKernelGGL(mnv_conv_bwd_bias_kernel<false>, dim3(top_num_channels, groups),
                       dim3(MNV_BIAS_THREADS), 0, s, top_diff, out, num_images, top_num_channels,
                       (int)hw, per);
  int rc = MNV_LAUNCH_STATUS();
  if (rc || groups == 1) return rc;
  hipLaunchKernelGGL(mnv_conv_bwd_bias_finish_kernel, dim3((top_num_channels + 3) / 4),
                     dim3(256), 0, s, reinterpret_cast<const float*>(workspace), bias_diff,
                     top_num_channels, groups);
  return MNV_LAUNCH_STATUS();
}

}  // extern "C"
