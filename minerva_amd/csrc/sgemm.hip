// SGEMM C{m,n} = A{m,k} * B{k,n}, column-major, no transposes, alpha 1 / beta 0:
// the product Minerva's MatMult asks for (reference minerva/op/impl/basic.cpp:150-173;
// cublasSgemm call at minerva/op/impl/cuda/cuda_perform.cu:66-70).
// Built on the matrix cores, in bf16 parts (gemm_split.h) for products of enough work and with the
// fp32 instruction (gemm_core.h) for the others; A is fetched x-fast (m contiguous), B k-fast (k
// contiguous).  Products with too few output tiles to fill 256 CUs split the k range over
// blockIdx.z when the caller lends a workspace.
#include <cmath>
#include <mutex>

#include "gemm_split.h"

// Split-k partial sums of mnv_sgemm_nn_static: one array per GPU the library is loaded on,
// held until the process ends.  In host code the name `scratch` is only a handle for
// hipGetSymbolAddress; kernels and every other use take the address it returns.
#define MNV_SGEMM_STATIC_SCRATCH_FLOATS ((size_t)MNV_SGEMM_STATIC_SCRATCH_BYTES / sizeof(float))
static __device__ __align__(256) float scratch[MNV_SGEMM_STATIC_SCRATCH_FLOATS];

namespace {

// Period 0 holds every full 16-deep slab: the per-thread byte offsets are fixed and only
// the uniform slab offset moves.  A k extent that is not a multiple of 16 leaves one
// partial slab, which is period 1 and gets its own masked offsets.
// TA / TB: the operand is given transposed -- A as {k,m} (element (m,k) at k + m*lda), B as
// {n,k} (element (k,n) at n + k*ldb) -- which only swaps its fetch direction: a transposed A
// is k-fast, a transposed B x-fast.  The values multiplied and the order they are added in
// are those of the product of the explicitly transposed matrices.
//
// Every vector is one 16-byte load whatever the extents and the alignment: buffer loads want
// 4-byte alignment only and check their range dword by dword.
//  x-fast: a vector that reaches past the last row (column) brings values of the next one;
//    they are summed into accumulators that are never stored.
//  k-fast: a vector that reaches past K brings values that would be summed.  K4 (K % 4 == 0):
//    there is none.  Otherwise the vectors of the last, partial slab are cleared past K on
//    their way to LDS (a_stash_fix, b_stash_fix: a uniform branch per slab; an infinity there
//    times the other operand's 0 would not be 0).
// Four 4-byte loads per vector, which odd extents took before, keep four times as many
// load instructions in a slab: 1001 x 250 x 4099 41.0 -> 28.5 us, 4099 x 4099 x 1023
// 292 -> 272, 10 x 256 x 256 9.4 -> 7.3; the same bits.  A transposed, in bf16 parts, where they also
// spill into the loop: 2230 x 2410 x 1302 173 -> 108 us, 2675 x 3691 x 237 64 -> 42 (fp32
// instruction 155 and 55).
template <bool K4, bool TA = false, bool TB = false>
struct SgemmNN {
  static constexpr bool A_KFAST = TA, B_KFAST = !TB;
  static constexpr int A_NOFF = 1, B_NOFF = 1;
  const float* __restrict__ A;
  const float* __restrict__ B;
  float* __restrict__ C;
  int M, N, K, total_slabs, spp, bk;
  // Leading dimensions (floats between consecutive columns as stored): m, k, m for whole
  // untransposed matrices (k for a transposed A, n for a transposed B); larger when the
  // operands are panels of matrices too large for 32-bit byte offsets.
  // accumulate: C += A*B (the k panels after the first).
  int lda, ldb, ldc, accumulate;
  // Fused epilogues (all off for the plain product), applied in this order to the value
  // stored, each the single operation the separate operator performs:
  //   bias: + bias[m] (the broadcast add of an {m,1} vector); relu: max(., 0);
  //   gate: gate[m,n] > 0 ? . : 0 (the ReLU gradient's selection)
  //   sgd_w (B transposed only, the weight gradient of an inner product): the value stored
  //   is sgd_w[m,n] - sgd_scale * ., the parameter update; C may be sgd_w itself
  const float* __restrict__ bias;
  const float* __restrict__ gate;
  int relu;
  const float* sgd_w;
  float sgd_scale;
  // Column tiles that are dealt m-tile by m-tile together, so that the 32 tiles an XCD works on
  // at a time are not all the rows of one column (see launch_split).
  static constexpr bool N_GROUPED = true;
  int n_group;
  struct Res {
    mnv_rsrc a, b;
  };
  struct AState {};
  struct BState {};
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(A, TA ? ((unsigned)(M - 1) * (unsigned)lda + (unsigned)K) * 4u
                              : ((unsigned)(K - 1) * (unsigned)lda + (unsigned)M) * 4u);
    r.b = mnv_make_rsrc(B, TB ? ((unsigned)(K - 1) * (unsigned)ldb + (unsigned)N) * 4u
                              : ((unsigned)(N - 1) * (unsigned)ldb + (unsigned)K) * 4u);
  }
  __device__ void a_init(const Res&, AState&, int) const {}
  __device__ void b_init(const Res&, BState&, int) const {}
  // A[m..m+3, k] (x-fast) or, transposed, A[m, k..k+3] (k-fast)
  __device__ void a_period(const AState&, unsigned (&off)[A_NOFF], int m, int kl, int period) const {
    const int k = period * spp * bk + kl;
    if (TA) {
      const unsigned base = ((unsigned)m * (unsigned)lda + (unsigned)k) * 4u;
#pragma unroll
      for (int q = 0; q < A_NOFF; ++q) off[q] = ((m < M) & (k < K)) ? base + 4u * q : MNV_OOB;
    } else {
      const unsigned base = ((unsigned)k * (unsigned)lda + (unsigned)m) * 4u;
#pragma unroll
      for (int q = 0; q < A_NOFF; ++q) off[q] = ((m < M) & (k < K)) ? base + 4u * q : MNV_OOB;
    }
  }
  __device__ void a_load(const Res& r, const AState&, const unsigned (&off)[A_NOFF], int, int s,
                         int, float (&v)[4]) const {
    mnv_fetch_vec<A_NOFF>(r.a, off, (unsigned)s * (unsigned)bk * (TA ? 1u : (unsigned)lda) * 4u, v);
  }
  // B[k..k+3, n] (k-fast) or, transposed, B[k, n..n+3] (x-fast)
  __device__ void b_period(const BState&, unsigned (&off)[B_NOFF], int n, int kl, int period) const {
    const int k = period * spp * bk + kl;
    if (TB) {
      const unsigned base = ((unsigned)k * (unsigned)ldb + (unsigned)n) * 4u;
#pragma unroll
      for (int q = 0; q < B_NOFF; ++q) off[q] = ((n < N) & (k < K)) ? base + 4u * q : MNV_OOB;
    } else {
      const unsigned base = ((unsigned)n * (unsigned)ldb + (unsigned)k) * 4u;
#pragma unroll
      for (int q = 0; q < B_NOFF; ++q) off[q] = ((n < N) & (k < K)) ? base + 4u * q : MNV_OOB;
    }
  }
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[B_NOFF], int, int s,
                         int, float (&v)[4]) const {
    mnv_fetch_vec<B_NOFF>(r.b, off, (unsigned)s * (unsigned)bk * (TB ? (unsigned)ldb : 1u) * 4u, v);
  }
  static constexpr bool A_STASH_FIX = !K4 && TA, B_STASH_FIX = !K4 && !TB;
  __device__ void a_stash_fix(int period, int s, int kl, float (&v)[4]) const { b_stash_fix(period, s, kl, v); }
  __device__ void b_stash_fix(int period, int, int kl, float (&v)[4]) const {
    if (period == (K >= bk ? 1 : 0)) {  // the partial slab
      const int rest = K % bk;
#pragma unroll
      for (int q = 1; q < 4; ++q) v[q] = kl + q < rest ? v[q] : 0.f;
    }
  }
  size_t extra_lds_bytes() const { return 0; }
  void set_bk(int b) {
    bk = b;
    spp = K >= b ? K / b : 1;
    total_slabs = (K + b - 1) / b;
  }
  __device__ void block_init(Res&, float*, int, int) const {}
  __device__ void c_store(int m, int n, float x) const {
    const size_t at = (size_t)n * ldc + m;
    if (accumulate) x = C[at] + x;
    if (bias) x = x + bias[m];
    if (relu) x = x > 0.f ? x : 0.f;
    if (gate) x = gate[at] > 0.f ? x : 0.f;
    if (TB) {
      if (sgd_w) x = sgd_w[at] - sgd_scale * x;
    }
    C[at] = x;
  }
  // four consecutive rows of one column: one 16-byte store for the plain product, element by
  // element when an epilogue is on
  static constexpr bool C_STORE4 = true;
  __device__ void c_store4(int m, int n, const float (&x)[4]) const {
    if (m + 3 < M && !accumulate && !bias && !relu && !gate && !sgd_w) {
      const mnv_f4u v = {x[0], x[1], x[2], x[3]};
      *reinterpret_cast<mnv_f4u*>(C + (size_t)n * ldc + m) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (m + q < M) c_store(m + q, n, x[q]);
    }
  }
  // the update read ahead of the block's stores (only bias / relu / gate / accumulate off)
  static constexpr bool C_PRELOAD = TB;
  __device__ bool c_preload_on() const { return sgd_w != nullptr; }
  __device__ float c_preload(int m, int n) const { return sgd_w[(size_t)n * ldc + m]; }
  __device__ void c_store_with(int m, int n, float x, float w) const {
    C[(size_t)n * ldc + m] = w - sgd_scale * x;
  }
};

// Products with at most 12 columns (inner products over a few images): every value of A is
// used that few times, so the product is bound by reading A once, while the smallest MFMA tile
// of the core multiplies 64 columns.  Here a lane keeps its four rows' sums for NC columns (N
// rounded up to one of a few widths; the columns past N repeat the last one and are not stored)
// and multiplies by B's values, which are the same for the whole wavefront and come through the
// scalar cache.  A load is 1 KB of a column.  A workgroup's four wavefronts take a quarter of its k
// range each, and their sums are added through LDS, (w0 + w2) + (w1 + w3); the k ranges of the
// grid's y dimension go through the workspace and the reduction kernel.
// Measured at 1 / 10 columns, with the reduction: 4096 x 9216 43.6 -> 26.4 us
// and 42.7 -> 33.2 us, 1000 x 4096 at 1 column 11.1 -> 6.6 us.
#define MNV_SKINNY_COLUMNS 12
template <class P, int NC, bool TB>
__global__ __launch_bounds__(256) void mnv_sgemm_skinny_kernel(P prob, const float* __restrict__ B, int k_per_wave,
                                                               float* __restrict__ partial) {
  constexpr int RM = 4, U = NC <= 4 ? 16 : NC <= 8 ? 8 : 4;  // rows per lane, k per step
  __shared__ float red[2 * MNV_WAVE * RM * NC];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / MNV_WAVE)), lane = threadIdx.x % MNV_WAVE;
  const int m = (blockIdx.x * MNV_WAVE + lane) * RM;
  int k = ((int)blockIdx.y * 4 + wave) * k_per_wave;
  const int k_end = k + k_per_wave < prob.K ? k + k_per_wave : prob.K;
  typename P::Res res;
  prob.make_res(res);
  // B's element (k, j), its address the same in every lane
  const int bk = TB ? prob.ldb : 1;
  size_t col[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) col[j] = (size_t)(j < prob.N ? j : prob.N - 1) * (TB ? 1 : prob.ldb);
  float acc[NC][RM];
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int q = 0; q < RM; ++q) acc[j][q] = 0.f;
  // bytes from the wavefront's k to the lane's rows; the rest of the address is uniform
  const unsigned off[1] = {m < prob.M ? (unsigned)m * 4u : MNV_OOB}, ak = (unsigned)prob.lda * 4u;
  auto step = [&](auto S, auto CUT) {
    constexpr int steps = decltype(S)::value;
    constexpr bool cut = decltype(CUT)::value;  // k + steps may pass k_end: 0 times -0 there, which leaves every sum as it is
    float v[steps][RM];
#pragma unroll
    for (int u = 0; u < steps; ++u) {
      const unsigned o[1] = {cut && k + u >= k_end ? MNV_OOB : off[0]};
      mnv_fetch_vec<1>(res.a, o, (unsigned)(k + u) * ak, v[u]);
    }
#pragma unroll
    for (int u = 0; u < steps; ++u)
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const bool on = !cut || k + u < k_end;
        const float x = B[col[j] + (size_t)(on ? k + u : k) * bk], b = on ? x : -0.f;
#pragma unroll
        for (int q = 0; q < RM; ++q) acc[j][q] = __builtin_fmaf(v[u][q], b, acc[j][q]);
      }
    k += steps;
  };
  typedef std::false_type Whole;
  while (k + U <= k_end) step(std::integral_constant<int, U>{}, Whole{});
  if (U > 8 && k + 8 <= k_end) step(std::integral_constant<int, 8>{}, Whole{});
  if (U > 4 && k + 4 <= k_end) step(std::integral_constant<int, 4>{}, Whole{});
  if (k < k_end) step(std::integral_constant<int, 4>{}, std::true_type{});
  auto put = [&](int region) {
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int q = 0; q < RM; ++q) red[((region * NC + j) * RM + q) * MNV_WAVE + lane] = acc[j][q];
  };
  auto add = [&](int region) {
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int q = 0; q < RM; ++q) acc[j][q] += red[((region * NC + j) * RM + q) * MNV_WAVE + lane];
  };
  if (wave >= 2) put(wave - 2);
  __syncthreads();
  if (wave < 2) add(wave);
  __syncthreads();
  if (wave == 1) put(0);
  __syncthreads();
  if (wave != 0) return;
  add(0);
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int q = 0; q < RM; ++q)
      if (j < prob.N && m + q < prob.M) {
        if (gridDim.y > 1) partial[((size_t)blockIdx.y * prob.N + j) * prob.M + m + q] = acc[j][q];
        else prob.c_store(m + q, j, acc[j][q]);
      }
}

// The same with A given transposed: every value added in the order of the kernel above, so that
// the bits are the same.  A row of A is contiguous along k, and a lane that walks its own row
// reads 16 bytes of a line per load, 64 lines at once (4096 x 4096 at 4 / 12 columns 25.8 / 92.8 us,
// where the tiles take 24.1 / 25.1; this kernel 16.7 / 18.0).  The workgroup's 64 rows and B's
// columns come in runs of RUN k instead, through an LDS strip of the wavefront's own (a wavefront's
// LDS accesses execute in order; the pitch spreads eight lanes' 16-byte reads over all banks), the
// next run in flight under the multiplies.  A value of B would then meet one row per lane, too
// few multiplies for a load from the scalar cache (24.7 / 55.5 us); the 16 x 16 x 1 and
// 4 x 4 x 1 matrix instructions add one k to all 64 rows and 16 or 4 columns, one multiply-add per
// element.  RUN: 128 bytes of a row, or 64 where a wavefront has no more than 16 k (half the
// LDS, twice the workgroups on a CU: 8192 x 1 x 512 10.4 -> 8.0 us).  Neighbouring workgroups take
// the k ranges of the same rows: with the row blocks first, a pitch that is a power of two keeps few memory
// channels busy (9216 x 1 x 4096 50.6 -> 34.2 us).
template <class P, int RUN, int COLS>
__global__ __launch_bounds__(256) void mnv_sgemm_skinny_tn_kernel(P prob, int k_per_wave, int ranges,
                                                                  float* __restrict__ partial) {
  constexpr int REGS = COLS;                               // of a lane's 64 x COLS / 64 sums
  typedef float Acc __attribute__((ext_vector_type(REGS)));
  constexpr int PITCH = RUN + 4, LPL = RUN / 4, PER = MNV_WAVE / LPL;  // lanes per line, lines per load
  constexpr int LINES = MNV_WAVE + (COLS > PER ? COLS : PER), VECS = LINES / PER, AV = MNV_WAVE / PER;  // A's rows, B's columns
  __shared__ __align__(16) float strips[4 * LINES * PITCH];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / MNV_WAVE)), lane = threadIdx.x % MNV_WAVE;
  const int range = (int)blockIdx.x % ranges, m0 = (int)blockIdx.x / ranges * MNV_WAVE;
  const int line = lane / LPL, k4 = lane % LPL * 4;
  int k = (range * 4 + wave) * k_per_wave;
  const int k_end = k + k_per_wave < prob.K ? k + k_per_wave : prob.K;
  typename P::Res res;
  prob.make_res(res);
  float* const strip = strips + wave * LINES * PITCH;
  // Rows past M and k past the last row's end lie past the tensor, where loads answer 0.  The
  // columns past N repeat the last one and are not stored.
  const unsigned pitch = (unsigned)prob.lda * 4u;
  float v[VECS][4];
  auto load = [&](int at) {
    const bool on = at + k4 < k_end;
#pragma unroll
    for (int u = 0; u < VECS; ++u) {
      const int j = (u - AV) * PER + line;
      const unsigned row = u < AV ? (unsigned)(m0 + line) * pitch : (unsigned)(j < prob.N ? j : prob.N - 1) * (unsigned)prob.ldb * 4u;
      const unsigned off[1] = {on ? row + (unsigned)k4 * 4u : MNV_OOB};
      mnv_fetch_vec<1>(u < AV ? res.a : res.b, off, (u < AV ? (unsigned)(u * PER) * pitch : 0u) + (unsigned)at * 4u, v[u]);
    }
  };
  Acc acc = 0.f;
  if (k < k_end) load(k);
  for (; k < k_end; k += RUN) {
    const int count = k_end - k < RUN ? k_end - k : RUN;
    if (count < RUN) {  // what lies past the range multiplies 0 by -0, which leaves every sum as it is
#pragma unroll
      for (int u = 0; u < VECS; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = k4 + e < count ? v[u][e] : u < AV ? 0.f : -0.f;
    }
#pragma unroll
    for (int u = 0; u < VECS; ++u)
      *reinterpret_cast<mnv_f4*>(strip + (u * PER + line) * PITCH + k4) = mnv_f4{v[u][0], v[u][1], v[u][2], v[u][3]};
    __builtin_amdgcn_wave_barrier();
    if (k + RUN < k_end) load(k + RUN);
    auto multiply = [&](int kk) {
      const mnv_f4 a = *reinterpret_cast<const mnv_f4*>(strip + lane * PITCH + kk);
      const mnv_f4 b = *reinterpret_cast<const mnv_f4*>(strip + (MNV_WAVE + lane % COLS) * PITCH + kk);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (COLS == 16) acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a[e], b[e], acc, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a[e], b[e], acc, 0, 0, 0);
      }
    };
    if (count == RUN) {
#pragma unroll
      for (int kk = 0; kk < RUN; kk += 4) multiply(kk);
    } else {
      for (int kk = 0; kk < count; kk += 4) multiply(kk);
    }
    __builtin_amdgcn_wave_barrier();
  }
  // Register q of lane l holds row q / 4 * 16 + l / 16 * 4 + q % 4 and column l % 16, or row l / 4 * 4 + q
  // and column l % 4; it lies at q * 65 + l of a region, neighbouring rows of a column in different banks.
  float* const red = strips;
  constexpr int REGION = REGS * 65;
  __syncthreads();  // the strips become the wavefronts' sums
  if (wave >= 2) {
#pragma unroll
    for (int q = 0; q < REGS; ++q) red[(wave - 2) * REGION + q * 65 + lane] = acc[q];
  }
  __syncthreads();
  if (wave < 2) {
#pragma unroll
    for (int q = 0; q < REGS; ++q) {
      float* at = red + wave * REGION + q * 65 + lane;
      *at = acc[q] + *at;
    }
  }
  __syncthreads();
  const int r = lane, m = m0 + r;
  if (m >= prob.M) return;
  for (int j = wave; j < prob.N; j += 4) {
    const float* at = red + (COLS == 16 ? (r / 16 * 4 + r % 4) * 65 + r % 16 / 4 * 16 : r % 4 * 65 + r / 4 * 4) + j;
    const float x = at[0] + at[REGION];
    if (ranges > 1) partial[((size_t)range * prob.N + j) * prob.M + m] = x;
    else prob.c_store(m, j, x);
  }
}

// Small products: T x T tiles (16 or 32) of the result, one per workgroup, whose W wavefronts share the k range.  A 64 x 64 tile
// of the core takes 0.24 us of a CU's matrix cores per 16 k and leaves most CUs without one; four or sixteen times as
// many tiles spread the same multiplies over them, and the k ranges meet in LDS, not in memory and a second launch.
// No operand passes through LDS: a lane loads what it multiplies, 16 bytes along k (a k-fast operand) or 4 bytes a k
// (x-fast, neighbouring lanes at neighbouring addresses), 32 k at a time, the next 32 in flight under the multiplies
// (96 in flight: no faster).  Of instruction t, lane group h (of 64 / T) takes k = 4 h + t of each run of 4 * 64 / T, in every
// form, so that the transposed forms have the bits of transposing first.  The wavefronts' sums are added in the order of k.
// k past K: an x-fast operand reads 0 past its end, a k-fast one is cleared; rows and columns past the result's may
// read anything inside the operand and are not stored.
// What bounds it: a launch and two trips to memory, 3 us; from one tile per CU on the operands' way from L2
// (128 or 256 bytes per k and tile).  An XCD works on neighbouring tiles across the shorter side of the result, so that its
// L2 fetches an eighth of the longer operand (4021 x 169 x 731 on 32 x 32 tiles 25 -> 17 us, 2093 x 198 x 3376 on 16 x 16 147 -> 55).
// us, tiles of the core -> this: 17 x 53 x 124 6.8 -> 3.1, 256 x 256 x 784 9.4 -> 4.3, 10 x 256 x 256 6.8 -> 3.3, 512 x 512 x 512
// 13.1 -> 5.9, 1421 x 284 x 488 14.4 -> 9.3, 1001 x 250 x 4099 29.3 -> 24.1; 283 random products of up to
// 4096 in every extent 0.59 of the time.
// Error against float64: a wavefront adds runs of 32 k up, each run under the next one's instructions, so that no sum is longer than
// 32 products or its own runs: 0.69 of the core's (of k ranges where it had them) over those 283 products of normal operands, none above
// 1.01 times; uniform ones 0.70, and 0.91 where both come from a ReLU (1.18 at most), whose zeros cost a plain sum nothing.
// With one sum each for the even and the odd fetches instead, 0.81 and up to 1.11, and 55 of the uniform products worse by up to 1.24;
// 1001 x 250 x 4099 2.99e-7 -> 1.54e-7, 25.3 us with the eight wavefronts that it then needed.
template <class P, int T, int W>
__global__ __launch_bounds__(W * MNV_WAVE, 4) void mnv_sgemm_small_kernel(P prob, int tiles_m, int tiles_n, int k_per_wave) {
  constexpr int H = MNV_WAVE / T, RUN = 4 * H, VECS = 32 / RUN, REGS = T * T / MNV_WAVE;
  typedef float Acc __attribute__((ext_vector_type(REGS)));
  __shared__ float red[W * T * T];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / MNV_WAVE)), lane = threadIdx.x % MNV_WAVE;
  const int x = lane % T, h = lane / T;
  const int tile = mnv_tile_remap((int)blockIdx.x, tiles_m * tiles_n);
  const bool tall = tiles_m > tiles_n;
  const int across = tall ? tiles_n : tiles_m, outer = tile / across, inner = tile - outer * across;
  const int m0 = (tall ? outer : inner) * T, n0 = (tall ? inner : outer) * T;
  typename P::Res res;
  prob.make_res(res);
  const unsigned lda = (unsigned)prob.lda * 4u, ldb = (unsigned)prob.ldb * 4u;
  const unsigned a_off = P::A_KFAST ? (m0 + x < prob.M ? (unsigned)(m0 + x) * lda + (unsigned)h * 16u : MNV_OOB)
                                    : (unsigned)h * 4u * lda + (unsigned)(m0 + x) * 4u;
  const unsigned b_off = P::B_KFAST ? (n0 + x < prob.N ? (unsigned)(n0 + x) * ldb + (unsigned)h * 16u : MNV_OOB)
                                    : (unsigned)h * 4u * ldb + (unsigned)(n0 + x) * 4u;
  auto fetch = [&](mnv_rsrc r, unsigned off, unsigned ld, auto KFAST, int k, float (&v)[VECS][4]) {
#pragma unroll
    for (int j = 0; j < VECS; ++j) {
      if constexpr (decltype(KFAST)::value) {
        const unsigned one[1] = {off};
        mnv_fetch_vec<1>(r, one, (unsigned)(k + RUN * j) * 4u, v[j]);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          v[j][t] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)((unsigned)(k + RUN * j + t) * ld), 0));
      }
    }
  };
  typedef std::integral_constant<bool, P::A_KFAST> AFast;
  typedef std::integral_constant<bool, P::B_KFAST> BFast;
  int k = wave * k_per_wave;
  const int k_end = k + k_per_wave < prob.K ? k + k_per_wave : prob.K;
  Acc sum = 0.f, run[2] = {0.f, 0.f};  // runs of 32 k
  float a[2][VECS][4], b[2][VECS][4];
  if (k < k_end) {
    fetch(res.a, a_off, lda, AFast{}, k, a[0]);
    fetch(res.b, b_off, ldb, BFast{}, k, b[0]);
  }
  auto step = [&](auto SET) {
    constexpr int set = decltype(SET)::value;
    fetch(res.a, a_off, lda, AFast{}, k + 32, a[set ^ 1]);  // past the range: not multiplied
    fetch(res.b, b_off, ldb, BFast{}, k + 32, b[set ^ 1]);
    if (k + 32 > prob.K) {
#pragma unroll
      for (int j = 0; j < VECS; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const bool on = k + RUN * j + 4 * h + t < prob.K;
          if (P::A_KFAST) a[set][j][t] = on ? a[set][j][t] : 0.f;
          if (P::B_KFAST) b[set][j][t] = on ? b[set][j][t] : 0.f;
        }
    }
#pragma unroll
    for (int j = 0; j < VECS; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const Acc before = j == 0 && t == 0 ? Acc(0.f) : run[set];
        if constexpr (T == 32) run[set] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[set][j][t], a[set][j][t], before, 0, 0, 0);
        else run[set] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[set][j][t], a[set][j][t], before, 0, 0, 0);
        if (j == 0 && t == 1) sum += run[set ^ 1];  // the run before, under this one's instructions
      }
    k += 32;
  };
  int steps = (k_end - k + 31) / 32;
  for (; steps >= 2; steps -= 2) {
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
  }
  if (steps > 0) {
    step(std::integral_constant<int, 0>{});
    sum += run[0];
  } else {
    sum += run[1];
  }
  // register r of lane (x, h): row x, column 4 h + r % 4 + 8 (r / 4)
#pragma unroll
  for (int r = 0; r < REGS; ++r) red[wave * T * T + (4 * h + r % 4 + 8 * (r / 4)) * T + x] = sum[r];
  __syncthreads();
  for (int e = threadIdx.x; e < T * T; e += W * MNV_WAVE) {
    float sum = red[e];
#pragma unroll
    for (int w = 1; w < W; ++w) sum += red[w * T * T + e];
    const int m = m0 + e % T, n = n0 + e / T;
    if (m < prob.M && n < prob.N) prob.c_store(m, n, sum);
  }
}

struct SgemmEpilogue {
  const float* bias;
  const float* gate;
  int relu;
  int lda = 0, ldb = 0, ldc = 0, accumulate = 0;  // 0: the matrices' own m, k, m
  const float* sgd_w = nullptr;
  float sgd_scale = 0.f;
};

template <bool K4, bool TA = false, bool TB = false>
SgemmNN<K4, TA, TB> make_sgemm(const float* a, const float* b, float* c, int m, int n, int k,
                                const SgemmEpilogue& e) {
  SgemmNN<K4, TA, TB> p;
  p.A = a; p.B = b; p.C = c; p.M = m; p.N = n; p.K = k;
  p.bias = e.bias; p.gate = e.gate; p.relu = e.relu;
  p.lda = e.lda ? e.lda : (TA ? k : m); p.ldb = e.ldb ? e.ldb : (TB ? n : k); p.ldc = e.ldc ? e.ldc : m;
  p.accumulate = e.accumulate;
  p.sgd_w = e.sgd_w; p.sgd_scale = e.sgd_scale;
  p.n_group = 1;
  p.set_bk(16);
  return p;
}

typedef MnvGemmTile<64, 64, 16, 2, 2> TileSmall;
typedef MnvGemmTile<128, 128, 16, 2, 2> TileBig;  // products of one slab (see plan_split)
// Of the bf16 parts: two workgroups per CU, one, and one with twice the rows.
typedef MnvSplitTile<128, 128, 2, 4, 1> SplitPair;
typedef MnvSplitTile<128, 128, 2, 4, 2> SplitOne;
typedef MnvSplitTile<256, 128, 4, 2, 2> SplitTall;
#define MNV_SGEMM_MAX_SPLITS 16
const long long kSmallOperand = (1LL << 29) - 1;  // floats that mnv_sgemm_small_kernel's offsets reach

// Tile shape and number of k ranges for an (m,n,k) product given `ws_floats` floats of
// scratch.  Both shapes are priced with the occupancy model of mnv_pick_splits, in units of
// one 128x128x16 slab: a 64x64 slab is a quarter of the arithmetic at about 80% of the
// efficiency, and every extra k range writes and re-reads m*n floats (about 1.2 us per
// slab unit, 6 TB/s for the partial sums).
struct SgemmPlan {
  bool small;
  int splits;
  int groups = 1;  // 4: workgroups of four wavefront groups that share a tile's k range
  bool tall = false;  // 256 x 128 tiles (no k ranges, one wavefront group)
  bool split = false; // in bf16 parts (256 x 128 tiles always, 128 x 128 ones but for a single slab)
  int skinny = 0;     // > 0: mnv_sgemm_skinny_kernel or, A transposed, its _tn_ twin; this many k per wavefront
  int tile = 0;       // 16, 32: mnv_sgemm_small_kernel with `groups` wavefronts
  double us = 0.0;    // the estimate of one on 64 x 64 or larger tiles
  bool from_grouped = false;  // in parts by plan_grouped
};

// Enough k ranges for 2048 wavefronts (eight on each CU, 4 KB or more of A in flight in each), with
// at least 16 k per wavefront, beyond 65 ranges 32 (1024 x 1 x 8192 12.2 -> 9.4 us).  The ranges are
// whole steps of 16 k: only the wavefront at the end of k meets the kernels' cut steps.
// The tiles stay for a small A, where the time is that of two launches either way, and for more
// columns, where the multiplies, not A's bytes, take this kernel's time; their own time does
// not change from 1 to 64 columns.  The transposed and fused forms share the plan, and their bits.
// Tiles -> this kernel, us, plain / B transposed / A transposed (* where the rule keeps the tiles):
//   4 columns: 512 x 1024 6.8 -> 6.7 / 6.8 -> 7.1 / 6.5 -> 6.2, 1000 x 1500 7.5 -> 7.3 / 7.8 -> 7.8 /
//     7.4 -> 6.3, 1000 x 4096 11.6 -> 7.5 / 12.6 -> 8.2 / 10.5 -> 6.3
//   8 columns: *1024 x 1024 6.9 -> 8.7 / 7.1 -> 9.3 / 6.8 -> 6.4, 256 x 4096 10.3 -> 8.7 / 11.2 -> 9.3 /
//     10.2 -> 6.4, *768 x 3000 9.2 -> 9.7 / 9.9 -> 10.2 / 9.2 -> 7.3, 2000 x 2000 10.1 -> 10.0 / 10.7 -> 10.6 /
//     9.9 -> 8.3, 4096 x 1000 10.3 -> 9.4 / 10.9 -> 10.0 / 10.2 -> 7.8; few k, so that a workgroup's start
//     and end weigh more: *40000 x 100 8.9 -> 9.6 / 9.3 -> 11.4 / 8.8 -> 5.4, *30000 x 150 9.8 -> 11.1 /
//     9.1 -> 11.6 / 10.2 -> 9.3, 100000 x 64 11.5 -> 9.7 / 11.7 -> 10.4 / 11.0 -> 6.3
//   12 columns: *4096 x 2048 15.0 -> 15.1 / 15.0 -> 16.5 / 14.8 -> 12.4, *1024 x 8192 15.2 -> 18.9 / 15.3 ->
//     19.4 / 15.2 -> 13.0, 4096 x 4096 24.5 -> 20.6 / 25.3 -> 24.0 / 23.7 -> 17.5, 1024 x 16384 23.1 -> 22.8 /
//     23.3 -> 25.2 / 24.0 -> 18.9, 9216 x 4096 45.4 -> 33.3 / 47.7 -> 40.9 / 44.5 -> 34.7
//   16 columns: *2000 x 2000 10.8 -> 16.9, *4096 x 4096 25.1 -> 25.4
// They also stay where the workspace holds fewer ranges and they make less than 128 workgroups, and
// below 256 rows (one block).
bool plan_skinny(int m, int n, int k, size_t ws_floats, SgemmPlan* plan) {
  const long long least = n <= 4 ? 1LL << 19 : n > 8 ? 1LL << 24 : k >= 4096 ? 1LL << 20 : k >= 256 ? 7LL << 19 : 3LL << 21;  // elements of A
  if (n > MNV_SKINNY_COLUMNS || m < 256 || k < 64 || (long long)m * k < least) return false;
  const int blocks = (m + 255) / 256;
  int per, ranges;
  auto cut = [&](long long splits) {
    per = (int)((k + 4 * splits - 1) / (4 * splits) + 15) / 16 * 16;
    ranges = (int)(((long long)k + 4LL * per - 1) / (4LL * per));
  };
  const int most = 512 / blocks;
  int slices = k < 128 ? 1 : (k + 63) / 64;
  if (slices > 65) slices = k > 65 * 128 ? (k + 127) / 128 : 65;
  cut(most < 1 ? 1 : most < slices ? most : slices);
  const size_t fit = ws_floats / ((size_t)m * n);
  if (ranges > 1 && (size_t)ranges > fit) {
    const long long have = fit ? (long long)fit : 1;  // one range needs no workspace
    if (blocks * have < 128) return false;
    cut(have);
  }
  *plan = SgemmPlan{false, ranges, 4};
  plan->skinny = per;
  return true;
}

// Microseconds of a product on 128 x 128 tiles in bf16 parts with z k ranges: a step of 32 k takes
// 1.13 where a CU has one workgroup (SplitOne), 1.3 of the CU's time for each where it has several
// (SplitPair); about 3 for a workgroup's first loads and last stores, 4 where up to three steps of
// a CU's one workgroup leave nothing to hide them behind (2871 x 1047 x 42 8.9 us with the fp32 instruction, 10.3 in parts; of 680 products of 36 to 700 k,
// 12 lost 7 to 16% to it with 3, 4 with 4, by up to 8%, and 3 gained that much less); 4 for the reduction of
// the k ranges beside its bytes.
double split_cost(int m, int n, int k, int z, int cus) {
  const long long tiles = (long long)((m + 127) / 128) * ((n + 127) / 128);
  const long long per_cu = (tiles * z + cus - 1) / cus;
  const int slabs = (k + 15) / 16, steps = ((slabs + z - 1) / z + 1) / 2;
  const double work = per_cu == 1 ? 1.13 * steps + (steps <= 3 ? 4.0 : 3.0) : 1.3 * per_cu * steps + 3.0 * (double)((per_cu + 1) / 2);
  return work + (z > 1 ? 4.0 + 8.0 * (double)m * n * z / 6e6 : 0.0);
}

// Which products run in bf16 parts.  Those planned on large tiles do, with the k ranges of their
// plan where it wants workgroups of four wavefront groups, one per CU, and otherwise with those that
// split_cost prefers.  Those planned on 64 x 64 tiles do where split_cost puts them at 90% of the
// plan's cost (in slabs of a 128 x 128 tile, about 0.83 us) or less.  64 x 64 tiles themselves stay with the
// fp32 instruction: the cut of their operands takes 4.3 vector instructions per matrix instruction.
// us, fp32 instruction -> bf16 parts (* where the rule keeps the former):
//   4096 x 4096 x 4096 941 -> 601, 4096 x 9216 x 256 161 -> 110, 4096 x 4096 x 256 69 -> 51,
//   4096 x 256 x 9216 156 -> 109, 9216 x 256 x 4096 165 -> 121, 2048 x 2048 x 2048 152 -> 88,
//   4096 x 1000 x 1000 76 -> 48, 4096 x 100 x 4096 47 -> 32, 200 x 3000 x 4000 67 -> 48, 1500 x 1500 x 1500
//   73 -> 56, 2100 x 2100 x 700 61 -> 56, *512 x 512 x 512 12.7 -> 13.6, *300 x 300 x 300 8.4 -> 10.8,
//   *256 x 256 x 784 9.2 -> 11.9, *700 x 1500 x 90 8.4 -> 8.7; of the grouped 64 x 64 tiles *1000 x 256 x 4096
//   24.7 -> 22.2, *4096 x 50 x 9216 51 -> 49, *4096 x 256 x 1000 21.7 -> 24.0.
void plan_split(int m, int n, int k, size_t ws_floats, double cost, int cus, SgemmPlan* plan) {
  if (plan->tall || (!plan->small && plan->groups == 4)) {
    plan->split = true;
    return;
  }
  if (plan->groups == 4 || m <= 64 || n <= 64) return;
  // One slab fills half of a step, and what such a product takes is the time of its stores, which the fp32 kernel, with
  // twice the workgroups per CU, spreads better (fp32 instruction / parts, us: k = 16 4096 x 4096 16.4 / 18.9, 4096 x 9216
  // 30.0 / 33.7, k = 17 20.4 / 18.3, 38.9 / 32.4).  Those planned on 64 x 64 tiles gain as little by parts as they lose.
  if (k <= 16 && !plan->small) return;
  const long long tiles = (long long)((m + 127) / 128) * ((n + 127) / 128);
  const size_t fit = ws_floats / ((size_t)m * n);
  const int slabs = (k + 15) / 16;
  int best_z = 1;
  double best = split_cost(m, n, k, 1, cus);
  for (int z = 2; z <= MNV_SGEMM_MAX_SPLITS && (size_t)z <= fit && slabs / z >= 8 && tiles < 2LL * cus; ++z) {
    const double c = split_cost(m, n, k, z, cus);
    if (c < 0.97 * best) {
      best = c;
      best_z = z;
    }
  }
  // k ranges of under 18 us lose to those of the 64 x 64 tiles (617 x 332 x 1746 15.7 -> 18.1, 122 x 1419 x
  // 1663 16.1 -> 17.9; above, 785 x 426 x 2236 25.5 -> 21.8, 541 x 1220 x 2092 37.9 -> 29.6).
  if (plan->small && (best > 0.9 * 0.83 * cost || (best_z > 1 && best < 18.0))) return;
  *plan = SgemmPlan{false, best_z};
  plan->split = true;
}

// Grouped 64 x 64 tiles against parts.  Their four wavefronts sum a quarter of a k range each, rounded at every k.  One chain in parts, rounded at
// every eighth, is nearer to float64 where signs are mixed (0.66 of the error), but of positive terms, whose sum grows with k, it is
// sqrt(2) times as far (2408 x 1161 x 2681 of uniform operands 2.03e-7 -> 2.86e-7, both from a ReLU 0.98e-7 -> 2.28e-7); with twice
// the ranges half of that.  So parts have at least twice the ranges of the grouped tiles.  Of 889 random products that leave them none is
// slower, they take 0.79 of the time, and of the error 0.37 for normal and 0.54 for uniform operands, none more than before (both from
// a ReLU 0.75, 1.10 at most).  us, and errors of normal and uniform operands in 1e-7: 341 x 3956 x 1002 45 -> 37 (2.9 -> 1.3, 1.13 -> 0.85),
// 2177 x 1155 x 3047 203 -> 114 (5.0 -> 1.6, 2.1 -> 0.83; in one chain 130, 3.4, 3.0), 3106 x 1474 x 2652 231 -> 162, 1340 x 599 x 3458 69 -> 48, 200 x 3319 x 2055
// 44 -> 33, 2048 x 300 x 3000 42.5 -> 39.5 (five ranges instead of three 35.7, uniform 0.73 -> 0.74).
// At most 16 tiles of 128 x 128, whose 16 ranges make no more workgroups than CUs, stay (*1000 x 256 x 4096 24.7 -> 22.2, *4096 x 256 x 1000
// 21.7 -> 24.0), ranges of under 20 us (3312 x 73 x 1235 15.0 -> 18.0, 143 x 2058 x 1764 19.6 -> 21.2), and grouped tiles of exactly one per CU, the
// plan that the inner products of 256 columns are documented to have (*4096 x 256 x 4096 74 -> 56).  The estimate of
// the grouped tiles is 20% low below 700 k, where two ranges have to gain 18% (1882 x 897 x 472 22.5 -> 26.9), and above 1200 k as
// much too high; ranges of under 40 us have to gain a tenth.
void plan_grouped(int m, int n, int k, size_t ws_floats, int cus, SgemmPlan* plan) {
  if (plan->groups != 4 || !plan->small || m <= 64 || n <= 64) return;
  const long long tiles = (long long)((m + 127) / 128) * ((n + 127) / 128);
  if (tiles * MNV_SGEMM_MAX_SPLITS <= cus || (plan->splits == 1 && (m + 63LL) / 64 * ((n + 63) / 64) == cus)) return;
  const size_t fit = ws_floats / ((size_t)m * n);
  const int slabs = (k + 15) / 16;
  int best_z = 0;
  double best = 1e30;
  for (int z = 2 * plan->splits; z <= MNV_SGEMM_MAX_SPLITS && (size_t)z <= fit && slabs / z >= 8; ++z) {
    const double c = split_cost(m, n, k, z, cus);
    if (c < best) {
      best = c;
      best_z = z;
    }
  }
  if (!best_z || best < 20.0) return;
  if (best > (best_z == 2 && slabs < 50 ? 0.82 : best < 40.0 ? 0.9 : 1.0) * plan->us) return;
  *plan = SgemmPlan{false, best_z};
  plan->split = plan->from_grouped = true;
  plan->us = best;
}

// The cheapest of the plans whose partial results fit `ws_floats`.  `cus`: the device's, asked for once per
// call, since the query takes about 0.05 us and the plans below weigh some fifty launches.
SgemmPlan plan_within(int m, int n, int k, size_t ws_floats, int cus) {
  const int slabs = (k + 15) / 16;
  const size_t mn = (size_t)m * n;
  const double per_split = 8.0 * (double)mn / 6e6 / 1.2;
  SgemmPlan best{false, 1};
  if (plan_skinny(m, n, k, ws_floats, &best)) return best;
  double best_cost = 0;
  for (int small = 0; small < 2; ++small) {
    const int bm = small ? 64 : 128;
    const long long tiles = (long long)((m + bm - 1) / bm) * ((n + bm - 1) / bm);
    int max_splits = MNV_SGEMM_MAX_SPLITS;
    if (max_splits > slabs / 4) max_splits = slabs / 4;
    const size_t fit = mn ? ws_floats / mn : 0;
    if ((size_t)max_splits > fit) max_splits = (int)fit;
    if (tiles >= 4LL * cus || slabs < 8) max_splits = 1;  // one per resident workgroup
    const double unit = small ? 0.31 : 1.0;
    double cost;
    const int splits = mnv_pick_splits(tiles, slabs, max_splits, cus, per_split / unit, &cost);
    cost *= unit;
    const bool forced = small ? (m <= 64 || n <= 64) : false;
    if (small == 0 || forced || cost < best_cost) {
      best = SgemmPlan{small != 0, splits};
      best_cost = cost;
    }
  }
  // Workgroups of four wavefront groups (one per CU for the large tile, two for the small
  // one): a step multiplies four slabs, one per group, and ends in about five slab times
  // for the prologue and the addition through LDS.  Measured on the inner products of the
  // AlexNet shape, back to back at sustained clocks: 4096x256x9216 0.190 -> 0.180 ms,
  // 4096x256x4096 0.100 -> 0.092 ms (64x64 tiles, no k ranges in memory at all),
  // 1000x256x4096 0.0304 -> 0.0278 ms, 4096x256x1000 0.031 -> 0.025 ms; 9216x256x4096, whose
  // 144 large tiles do not divide the 256 CUs, stays with single groups.
  // The launch of the reduction kernel itself (about six slab times) only matters in this
  // comparison, where a plan without k ranges in memory competes.
  const double reduce_launch = 6.0;
  if (best.splits > 1) best_cost += reduce_launch;
  for (int small = 0; small < 2; ++small) {
    if (!small && (m <= 64 || n <= 64)) continue;
    const int bm = small ? 64 : 128;
    const long long tiles = (long long)((m + bm - 1) / bm) * ((n + bm - 1) / bm);
    const double unit = small ? 0.27 : 1.0, overhead = small ? 4.0 : 5.0;
    const size_t fit = mn ? ws_floats / mn : 0;
    for (int z = 1; z <= MNV_SGEMM_MAX_SPLITS; ++z) {
      if (z > 1 && (size_t)z > fit) break;
      const int len4 = ((slabs + z - 1) / z + 3) / 4;
      if (len4 < 8) break;  // shorter loops do not repay the prologue and the addition
      // The sixteen wavefronts of such a workgroup share every barrier, so each step waits
      // out a trip to memory that separate workgroups would overlap: worth it only when the
      // workgroups cover most of the chip (MLP 784-256-10 at batch 256, 16 tiles: 0.111 ms
      // per step with single groups, 0.158 ms with grouped ones).
      if (tiles * z < 192) continue;
      const long long per_cu = (tiles * z + 255) / 256;
      const double cost = (double)per_cu * (4.0 * len4 * unit + overhead) +
                          (z > 1 ? per_split * z + reduce_launch : 0.0);
      if (cost < best_cost * 0.95) {
        best = SgemmPlan{small != 0, z, 4};
        best_cost = cost;
      }
    }
  }
  // Large products whose 256 x 128 tiles fill the chip's two-per-CU slots in whole rounds
  // (at least 95% of the multiplies of all rounds are the product's own).  Every element is summed
  // over k in the same order as on the 128 x 128 tile: the same bits.  us on 128 x 128 / 256 x 128, plain, A
  // and B transposed: 4096^3 686 / 651, 681 / 623, 657 / 598; 4096 x 4096 x 512 91 / 90, 94 / 91, 89 / 87; 2048 x 8192 x
  // 1024 175 / 163, 178 / 166, 171 / 160.
  if (!best.small && best.splits == 1 && best.groups == 1 && m >= 256 && slabs >= 32) {
    const long long tiles = (long long)((m + 255) / 256) * ((n + 127) / 128);
    const long long slots = 2LL * cus, rounds = (tiles + slots - 1) / slots;
    if ((double)m * n >= 0.95 * (double)(rounds * slots) * 256.0 * 128.0) best.tall = true;
  }
  plan_split(m, n, k, ws_floats, best_cost, cus, &best);
  // in us, fitted to 500 random products of up to 3 GFLOP (10% off, rms)
  best.us = best.split ? split_cost(m, n, k, best.splits, cus) : best.groups == 4 ? (k % 4 ? 0.92 : 0.84) * best_cost : 0.77 * best_cost + 0.5;
  return best;
}

// A plan on the small kernel's tiles where that is estimated at less than 90% of `plan`: 3 us, and the larger of what the
// fullest CU multiplies and what all tiles take from L2, 1.49 and 1.95 us per 1000 k of a 16 x 16 tile on every CU, 4.36 and
// 4.81 of a 32 x 32 one (5.2 from 2048 k on); beyond the eight or four and a half workgroups per CU, 2.5 or
// 3.4 us for each further round (with 2.5 and five of the larger tiles: 555 x 2773 x 156 10.0 -> 11.6, 2411 x 630 x 201 12.6 -> 15.0, 433 x 3053 x 133
// 10.4 -> 11.4, 3921 x 332 x 232 13.0 -> 13.9, which now stay; 1770 x 721 x 430 25.6 -> 20.1 does not).
// Up to 128 k a round costs what it did with 2.5 and five workgroups: there the tiles of the core take longer than their estimate (864 x 1196 x 89
// 8.1 -> 6.3, 1752 x 632 x 126 9.2 -> 7.2).
// From 2048 k on 16 x 16 tiles take up to 1.4 times their estimate (292 x 243 x 3361 14.8 -> 21.7; 49 x 98 x 3847 11.7 -> 9.8) and are
// left to the k ranges; from 1024 k on those of more than four to a CU do, and count 2.6 us (509 x 513 x 1935 on tiles of the core 21.4, on these 30.0;
// 2468 x 102 x 1441 18.6, 21.4, on 32 x 32 tiles 18.4; 674 random products that leave them 0.90 of the time).  500 random products that it moves 0.56 of the time, none slower; 400 of at least 250 rows
// and columns 0.66, two slower by more than 3% (1538 x 609 x 248 9.9 -> 10.5, 459 x 1917 x 200 8.8 -> 9.2).  Four wavefronts for many tiles, eight for few.
// The kernel reads an x-fast operand up to 95 k past its end: its offsets have to stay below 2^31.
void plan_small(int m, int n, int k, int cus, SgemmPlan* plan) {
  // (other products in parts are the more exact ones)
  if (plan->skinny || (plan->split && !plan->from_grouped) || (k + 96LL) * m > kSmallOperand || (k + 96LL) * n > kSmallOperand) return;
  auto cost = [&](int t, double own, double all) {
    const double per_cu = (double)((m + t - 1LL) / t) * ((n + t - 1) / t) / cus;
    const double work = all * per_cu > own * ceil(per_cu) ? all * per_cu : own * ceil(per_cu);
    const double rounds = t == 16 ? 2.5 * (per_cu / 8.0 - 1.0) : k <= 128 ? 2.5 * (per_cu / 5.0 - 1.0) : 3.4 * (ceil(per_cu / 4.5) - 1.0);
    return 3.0 + work * 1e-3 * k + (rounds > 0.0 ? rounds : 0.0);
  };
  const bool fifth = k > 1024 && (m + 15LL) / 16 * ((n + 15) / 16) > 4LL * cus;
  const double c16 = k <= 2048 ? cost(16, 1.49, fifth ? 2.6 : 1.95) : 1e30, c32 = cost(32, k > 2048 ? 5.2 : 4.36, k > 2048 ? 5.2 : 4.81);
  if ((c16 < c32 ? c16 : c32) >= 0.9 * plan->us) return;
  *plan = SgemmPlan{true, 1};
  plan->tile = c16 < c32 ? 16 : 32;
  const bool many = plan->tile == 16 ? (long long)m * n > 512 * cus : (m + 31LL) / 32 * ((n + 31) / 32) >= cus;
  plan->groups = many ? 4 : 8;
}

// The plan of an unlimited workspace.  A plan is planned again within what its own partial results need,
// until that changes nothing: alternatives with more k ranges have then lost them.  A plan in bf16
// parts with k ranges stands, it won against the best that the others can be; one without has so far won
// against k ranges only, whose reduction costs short products more than they gain: 307 x 270 x 143 takes
// 7.5 us on 64 x 64 tiles without ranges, 8.3 with two, 12.5 in parts, 3059 x 183 x 194 9.2, 14.2 and 15.0.
// It stands too where grouped tiles would take its place, which plan_split has not weighed against it.
SgemmPlan plan_unlimited(int m, int n, int k, int cus) {
  SgemmPlan plan = plan_within(m, n, k, (size_t)-1, cus);
  while (!plan.split || (plan.splits == 1 && plan.groups == 1 && !plan.tall)) {
    const SgemmPlan next = plan_within(m, n, k, plan.splits > 1 ? (size_t)plan.splits * m * n : 0, cus);
    if (plan.split && next.groups == 4) break;
    const bool same = next.split == plan.split && next.small == plan.small && next.splits == plan.splits && next.groups == plan.groups;
    plan = next;
    if (same) break;
  }
  plan_grouped(m, n, k, (size_t)-1, cus, &plan);
  plan_small(m, n, k, cus, &plan);
  return plan;
}

// The plan of an unlimited workspace wherever its own partial results fit, so that the bytes the
// query asks for give the plan that the query was made for.  Planned within those bytes
// instead, the plans that lost against it would have fewer k ranges, one of them would win, and 1500 x
// 1500 x 1501 would stay on grouped 64 x 64 tiles (72 us with a large workspace, 88 with the queried one).
SgemmPlan plan_sgemm(int m, int n, int k, size_t ws_floats) {
  const int cus = mnv_cu_count();
  SgemmPlan plan = plan_unlimited(m, n, k, cus);
  if (plan.splits == 1 || plan.splits <= ws_floats / ((size_t)m * n)) return plan;
  plan = plan_within(m, n, k, ws_floats, cus);
  plan_grouped(m, n, k, ws_floats, cus, &plan);
  plan_small(m, n, k, cus, &plan);
  return plan;
}

template <int NC, bool TB, class P>
void launch_skinny(const SgemmPlan& plan, const P& p, float* part, hipStream_t s) {
  hipLaunchKernelGGL((mnv_sgemm_skinny_kernel<P, NC, TB>), dim3((p.M + 4 * MNV_WAVE - 1) / (4 * MNV_WAVE), plan.splits),
                     dim3(256), 0, s, p, p.B, plan.skinny, part);
}

template <int RUN, int COLS, class P>
void launch_skinny_tn(const SgemmPlan& plan, const P& p, float* part, hipStream_t s) {
  hipLaunchKernelGGL((mnv_sgemm_skinny_tn_kernel<P, RUN, COLS>), dim3((p.M + MNV_WAVE - 1) / MNV_WAVE * plan.splits),
                     dim3(256), 0, s, p, plan.skinny, plan.splits, part);
}

template <bool K4, bool TA, bool TB>
int launch_skinny_columns(const SgemmPlan& plan, const SgemmNN<K4, TA, TB>& p, void* workspace, hipStream_t s) {
  static_assert(!(TA && TB), "one operand transposed at most");
  float* part = plan.splits > 1 ? reinterpret_cast<float*>(workspace) : nullptr;
  if constexpr (TA) {
    if (p.N <= 4) {
      if (plan.skinny <= 16) launch_skinny_tn<16, 4>(plan, p, part, s);
      else launch_skinny_tn<32, 4>(plan, p, part, s);
    } else {
      if (plan.skinny <= 16) launch_skinny_tn<16, 16>(plan, p, part, s);
      else launch_skinny_tn<32, 16>(plan, p, part, s);
    }
  } else if (p.N <= 1) launch_skinny<1, TB>(plan, p, part, s);
  else if (p.N <= 2) launch_skinny<2, TB>(plan, p, part, s);
  else if (p.N <= 4) launch_skinny<4, TB>(plan, p, part, s);
  else if (p.N <= 8) launch_skinny<8, TB>(plan, p, part, s);
  else launch_skinny<MNV_SKINNY_COLUMNS, TB>(plan, p, part, s);
  const int rc = MNV_LAUNCH_STATUS();
  if (rc || plan.splits == 1) return rc;
  return mnv_gemm_reduce_launch(p, part, plan.splits, s);
}

template <int T, int W, class P>
int launch_small(const P& p, hipStream_t s) {
  const int tiles_m = (p.M + T - 1) / T, tiles_n = (p.N + T - 1) / T;
  hipLaunchKernelGGL((mnv_sgemm_small_kernel<P, T, W>), dim3(tiles_m * tiles_n), dim3(W * MNV_WAVE), 0, s, p, tiles_m, tiles_n,
                     (p.K + 32 * W - 1) / (32 * W) * 32);
  return MNV_LAUNCH_STATUS();
}

template <bool TA, bool TB>
int launch_small_tiles(const SgemmPlan& plan, const SgemmNN<true, TA, TB>& p, hipStream_t s) {
  if (plan.tile == 16) return plan.groups == 4 ? launch_small<16, 4>(p, s) : launch_small<16, 8>(p, s);
  return plan.groups == 4 ? launch_small<32, 4>(p, s) : launch_small<32, 8>(p, s);
}

// In bf16 parts.  Groups of up to eight column tiles, as many as divide them: 4096^3 on 256 x 128
// tiles reads 12 panels for 32 tiles where whole columns read 18.
template <class P>
int launch_split(const SgemmPlan& plan, P p, void* workspace, size_t tail_bytes, hipStream_t s) {
  const int tiles_n = (p.N + 127) / 128;
  while (p.n_group < 8 && tiles_n % (2 * p.n_group) == 0) p.n_group *= 2;
  if (plan.tall) return mnv_gemm_launch<SplitTall>(p, 1, workspace, s);
  const long long tiles = (long long)((p.M + 127) / 128) * tiles_n;
  return tiles * plan.splits <= mnv_cu_count() ? mnv_gemm_launch<SplitOne>(p, plan.splits, workspace, s)
                                               : mnv_gemm_launch<SplitPair>(p, plan.splits, workspace, s, tail_bytes);
}

// A launch without k ranges may use the workspace for the partial tiles of a cut tail.
template <class P>
int launch_plan(const SgemmPlan& plan, const P& p, void* workspace, size_t workspace_bytes,
                hipStream_t s) {
  const size_t tail_bytes = plan.splits == 1 && workspace ? workspace_bytes : 0;
  if (plan.split) return launch_split(plan, p, workspace, tail_bytes, s);
  if (plan.groups == 4) return mnv_gemm_launch<TileSmall, 4>(p, plan.splits, workspace, s);
  return plan.small ? mnv_gemm_launch<TileSmall>(p, plan.splits, workspace, s, tail_bytes)
                    : mnv_gemm_launch<TileBig>(p, plan.splits, workspace, s, tail_bytes);
}

// Bytes a product without k ranges wants for the partial tiles of its cut tail.
size_t sgemm_tail_bytes(const SgemmPlan& plan, int m, int n, int k) {
  if (plan.splits != 1 || plan.groups != 1 || plan.tall || plan.tile) return 0;
  const int bm = plan.small ? 64 : 128;
  const long long tiles = (long long)((m + bm - 1) / bm) * ((n + bm - 1) / bm);
  const MnvTailPlan t = mnv_tail_plan(tiles, (k + 15) / 16, (size_t)bm * bm, (size_t)-1 / sizeof(float),
                                      plan.split ? SplitPair::TAIL : MnvTailCost{});
  return t.z > 1 ? (size_t)(tiles - t.begin) * t.z * bm * bm * sizeof(float) : 0;
}

#define MNV_MAX_DEVICES 64
std::mutex g_scratch_mutex;
float* g_scratch_ptr[MNV_MAX_DEVICES];  // device address of `scratch` on each GPU

// The address of the current device's copy of `scratch`, looked up once per device.
int scratch_address(float** out) {
  int dev = -1;
  MNV_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= MNV_MAX_DEVICES) return MNV_ERR_INVALID;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    MNV_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return MNV_ERR_INVALID;
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = g_scratch_ptr[dev];
  return MNV_OK;
}

int sgemm_nn_impl(const float* a, const float* b, float* c, int m, int n, int k, void* workspace,
                  size_t workspace_bytes, hipStream_t s,
                  const SgemmEpilogue& e = SgemmEpilogue{nullptr, nullptr, 0}) {
  // a panel of larger matrices has their pitches, which the small kernel's reach is not planned for
  const SgemmPlan plan = e.lda ? plan_within(m, n, k, 0, mnv_cu_count()) : plan_sgemm(m, n, k, workspace ? workspace_bytes / sizeof(float) : 0);
  if (plan.skinny) return launch_skinny_columns(plan, make_sgemm<true>(a, b, c, m, n, k, e), workspace, s);
  if (plan.tile) return launch_small_tiles(plan, make_sgemm<true>(a, b, c, m, n, k, e), s);
  if (k % 4 == 0) return launch_plan(plan, make_sgemm<true>(a, b, c, m, n, k, e), workspace, workspace_bytes, s);
  return launch_plan(plan, make_sgemm<false>(a, b, c, m, n, k, e), workspace, workspace_bytes, s);
}

// Products with one operand given transposed: same plan (tile shape, k ranges) as the plain
// product of the same extents, so that the result has the bits of transposing first.
template <bool TA, bool TB>
int sgemm_t_impl(const float* a, const float* b, float* c, int m, int n, int k, void* workspace,
                 size_t workspace_bytes, hipStream_t s, const SgemmEpilogue& e) {
  const SgemmPlan plan = plan_sgemm(m, n, k, workspace ? workspace_bytes / sizeof(float) : 0);
  if (plan.skinny) return launch_skinny_columns(plan, make_sgemm<true, TA, TB>(a, b, c, m, n, k, e), workspace, s);
  if (plan.tile) return launch_small_tiles(plan, make_sgemm<true, TA, TB>(a, b, c, m, n, k, e), s);
  // with both operands x-fast no vector runs along k
  if ((!TA && TB) || k % 4 == 0)
    return launch_plan(plan, make_sgemm<true, TA, TB>(a, b, c, m, n, k, e), workspace, workspace_bytes, s);
  return launch_plan(plan, make_sgemm<false, TA, TB>(a, b, c, m, n, k, e), workspace, workspace_bytes, s);
}

// Operands of 2^29 elements and more (up to the reference's limit, int element counts): the
// product is cut into panels whose spans fit 32-bit byte offsets -- columns of B and C, rows
// of A and C, and ranges of k, the later k ranges accumulating into C -- each panel one launch
// with the whole matrices' leading dimensions.  Slower than one launch (C is re-read per k
// range, no k ranges over workgroups), and the sum over k is taken range by range.
const long long kOperandLimit = (1LL << 29) - 1;  // elements a launch can address per operand

bool sgemm_is_large(int m, int n, int k) {
  return (long long)m * k > kOperandLimit || (long long)k * n > kOperandLimit;
}

int sgemm_nn_large(const float* a, const float* b, float* c, int m, int n, int k, hipStream_t s) {
  const long long mc = m < (1 << 28) ? m : (1 << 28);
  long long kc = (kOperandLimit - mc) / m + 1;          // ((kc-1)*m + mc) <= limit
  if (kc > k) kc = k;
  if (kc >= 16) kc -= kc % 16;
  long long nc = (kOperandLimit - kc) / k + 1;          // ((nc-1)*k + kc) <= limit
  if (nc > n) nc = n;
  if (kc < 1 || nc < 1) return MNV_ERR_INVALID;
  for (long long n0 = 0; n0 < n; n0 += nc)
    for (long long m0 = 0; m0 < m; m0 += mc)
      for (long long k0 = 0; k0 < k; k0 += kc) {
        const int mm = (int)(m - m0 < mc ? m - m0 : mc), nn = (int)(n - n0 < nc ? n - n0 : nc);
        const int kk = (int)(k - k0 < kc ? k - k0 : kc);
        SgemmEpilogue e{nullptr, nullptr, 0, m, k, m, k0 > 0};
        int rc = sgemm_nn_impl(a + (size_t)k0 * m + m0, b + (size_t)n0 * k + k0,
                               c + (size_t)n0 * m + m0, mm, nn, kk, nullptr, 0, s, e);
        if (rc) return rc;
      }
  return MNV_OK;
}

}  // namespace

extern "C" {

size_t mnv_sgemm_nn_workspace_bytes(int m, int n, int k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  const SgemmPlan plan = plan_unlimited(m, n, k, mnv_cu_count());
  return plan.splits > 1 ? (size_t)plan.splits * m * n * sizeof(float) : sgemm_tail_bytes(plan, m, n, k);
}

int mnv_sgemm_nn_plan(int m, int n, int k, size_t workspace_bytes, int* tile_rows, int* k_ranges,
                      int* groups) {
  if (m <= 0 || n <= 0 || k <= 0 || !tile_rows || !k_ranges || !groups) return MNV_ERR_INVALID;
  const SgemmPlan plan = plan_sgemm(m, n, k, workspace_bytes / sizeof(float));
  *tile_rows = plan.tall || plan.skinny ? 256 : plan.small ? 64 : 128;
  const int slabs = (k + 15) / 16, per = (slabs + plan.splits - 1) / plan.splits;
  *k_ranges = plan.skinny ? plan.splits : (slabs + per - 1) / per;  // as the launch rounds it: ranges of equal length
  *groups = plan.tile ? 1 : plan.groups;
  return MNV_OK;
}

int mnv_sgemm_nn_small_plan(int m, int n, int k, size_t workspace_bytes, int* tile_rows, int* wavefronts) {
  if (m <= 0 || n <= 0 || k <= 0 || !tile_rows || !wavefronts) return MNV_ERR_INVALID;
  const SgemmPlan plan = plan_sgemm(m, n, k, workspace_bytes / sizeof(float));
  *tile_rows = plan.tile;
  *wavefronts = plan.tile ? plan.groups : 0;
  return MNV_OK;
}

int mnv_sgemm_nn(const float* a, const float* b, float* c, int m, int n, int k, void* workspace,
                 size_t workspace_bytes, mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!a || !b || !c || m < 0 || n < 0 || k <= 0) return MNV_ERR_INVALID;
  // every operand is at most 2^31 - 1 elements (the reference's int element counts)
  if ((long long)m * k > 0x7fffffffLL || (long long)k * n > 0x7fffffffLL ||
      (long long)m * n > 0x7fffffffLL)
    return MNV_ERR_INVALID;
  if (sgemm_is_large(m, n, k)) return sgemm_nn_large(a, b, c, m, n, k, mnv_stream(stream));
  return sgemm_nn_impl(a, b, c, m, n, k, workspace, workspace_bytes, mnv_stream(stream));
}

int mnv_sgemm_nn_bias(const float* a, const float* b, const float* bias, float* c, int m, int n,
                      int k, int relu, void* workspace, size_t workspace_bytes,
                      mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!a || !b || !bias || !c || m < 0 || n < 0 || k <= 0) return MNV_ERR_INVALID;
  if ((long long)m * k >= (1LL << 29) || (long long)k * n >= (1LL << 29)) return MNV_ERR_INVALID;
  return sgemm_nn_impl(a, b, c, m, n, k, workspace, workspace_bytes, mnv_stream(stream),
                       SgemmEpilogue{bias, nullptr, relu != 0});
}

int mnv_sgemm_nn_relu_bwd(const float* a, const float* b, const float* bottom, float* c, int m,
                          int n, int k, void* workspace, size_t workspace_bytes,
                          mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!a || !b || !bottom || !c || m < 0 || n < 0 || k <= 0) return MNV_ERR_INVALID;
  if ((long long)m * k >= (1LL << 29) || (long long)k * n >= (1LL << 29)) return MNV_ERR_INVALID;
  return sgemm_nn_impl(a, b, c, m, n, k, workspace, workspace_bytes, mnv_stream(stream),
                       SgemmEpilogue{nullptr, bottom, 0});
}

int mnv_sgemm_tn(const float* at, const float* b, const float* gate, float* c, int m, int n, int k,
                 void* workspace, size_t workspace_bytes, mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!at || !b || !c || m < 0 || n < 0 || k <= 0) return MNV_ERR_INVALID;
  if ((long long)m * k >= (1LL << 29) || (long long)k * n >= (1LL << 29)) return MNV_ERR_INVALID;
  return sgemm_t_impl<true, false>(at, b, c, m, n, k, workspace, workspace_bytes, mnv_stream(stream),
                                   SgemmEpilogue{nullptr, gate, 0});
}

int mnv_sgemm_nt(const float* a, const float* bt, float* c, int m, int n, int k, void* workspace,
                 size_t workspace_bytes, mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!a || !bt || !c || m < 0 || n < 0 || k <= 0) return MNV_ERR_INVALID;
  if ((long long)m * k >= (1LL << 29) || (long long)k * n >= (1LL << 29)) return MNV_ERR_INVALID;
  return sgemm_t_impl<false, true>(a, bt, c, m, n, k, workspace, workspace_bytes, mnv_stream(stream),
                                   SgemmEpilogue{nullptr, nullptr, 0});
}

int mnv_sgemm_nt_sgd(const float* a, const float* bt, const float* w, float scale, float* w_out,
                     int m, int n, int k, void* workspace, size_t workspace_bytes,
                     mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!a || !bt || !w || !w_out || m < 0 || n < 0 || k <= 0) return MNV_ERR_INVALID;
  if ((long long)m * k >= (1LL << 29) || (long long)k * n >= (1LL << 29)) return MNV_ERR_INVALID;
  SgemmEpilogue e{nullptr, nullptr, 0};
  e.sgd_w = w;
  e.sgd_scale = scale;
  return sgemm_t_impl<false, true>(a, bt, w_out, m, n, k, workspace, workspace_bytes,
                                   mnv_stream(stream), e);
}

int mnv_sgemm_nn_static(const float* a, const float* b, float* c, int m, int n, int k,
                        mnv_stream_t stream) {
  if (m == 0 || n == 0) return MNV_OK;
  if (!a || !b || !c || m < 0 || n < 0 || k <= 0) return MNV_ERR_INVALID;
  if ((long long)m * k >= (1LL << 29) || (long long)k * n >= (1LL << 29)) return MNV_ERR_INVALID;
  // at least two k ranges of partial sums must fit the static array
  if ((unsigned long long)m * (unsigned long long)n * 2ull > MNV_SGEMM_STATIC_SCRATCH_FLOATS)
    return MNV_ERR_TOO_LARGE;
  float* ws = nullptr;
  int rc = scratch_address(&ws);
  if (rc) return rc;
  return sgemm_nn_impl(a, b, c, m, n, k, ws, MNV_SGEMM_STATIC_SCRATCH_BYTES, mnv_stream(stream));
}

}  // extern "C"
