// fp32 products on the bf16 matrix cores of gfx950, with fewer roundings than on the fp32 ones.
//
// A value x is cut into three bf16 numbers, x = x1 + x2 + x3 with |x2| <= 2^-8 |x| and
// |x3| <= 2^-17 |x|; their 3 x 8 significant bits hold all 24 of x.  A product a b is then
//   a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1)
// and three terms of at most 2^-25 |a b| each that are left out (with all nine the error against
// float64 is the same to three digits).  The bf16 matrix instruction multiplies exactly and adds
// in fp32, 16 times as many products per cycle as the fp32 one, so that six of them per product
// still leave 2.6 times its rate.  What either instruction loses is the rounding of the running
// sum.  The fp32 one rounds at every k; the 16 x 16 x 32 bf16 one at every 8 (measured).  a1 b1
// has accumulators of its own, the five smaller terms, at 2^-8 of its size, another set: one
// rounding of the full sum for 8 k.  Error against float64 (2-norm, relative), fp32 instruction /
// this: k = 32 1.0e-7 / 0.4e-7, 576 4.3e-7 / 1.4e-7, 4096 11.3e-7 / 4.0e-7; with a left operand
// from a ReLU, whose zeros cost the fp32 sum nothing, 4096 8.3e-7 / 3.2e-7.  (One set of
// accumulators for all six: 9.9e-7 and 9.6e-7, the second worse than the fp32 instruction.)  Two kinds of
// sums gain nothing.  One of a single term (a one-hot or diagonal operand) is within 2^-23 and not
// 2^-24 of it, for the three terms left out (rms 2.53e-8 / 2.60e-8; 0 and 1 times a value stay exact).  One
// of positive terms only, where the fp32 kernel had four wavefronts sum a quarter of the k each: uniform
// operands 4096^3 8.4e-7 / 3.0e-7 (one chain), 2048^3 1.6e-7 / 2.2e-7, 3837 x 2065 x 4394 2.4e-7 / 3.4e-7 (both from a
// ReLU 1.3e-7 / 3.3e-7).  Folding the sums every 512 k into a third set of accumulators mends half of these
// (of 70 random extents of uniform operands 21 were worse than the fp32 kernel, and 10 with it): only one workgroup per
// CU leaves registers for it, and it costs up to 9% (1215 x 1372 x 3540 81 -> 88 us).  More k ranges mend it, and where the small
// tiles' four wavefronts are left for parts there are enough of them (plan_grouped).
//
// Range.  Operands are multiplied by 2^16 before the cut, so that the last bit of the smallest
// denormal is still a bf16 denormal, and the product by 2^-32 after the sum.  An operand from
// 2^111 on, or an infinity or NaN, makes x2 an infinity or a NaN where fp32 arithmetic may have
// a finite or an infinite result (inf * 1: 1 = 1 + 0 + 0, and inf * 0 is NaN), and a
// running sum from 2^96 on overflows: a wavefront whose sums are not all finite multiplies its block
// again with the fp32 instruction.
//
// Data path: HBM -> registers (the policies' fetches, gemm_core.h) -> cut -> three bf16 planes
// in LDS -> v_mfma_f32_16x16x32_bf16.  A step of the main loop is two 16-deep slabs of the
// policy; the first half of the wavefronts fetches and cuts the even slab, the second the odd
// one.  LDS holds 8-byte groups of four consecutive k of one x, plane by plane, [k / 4][position of x]; a
// k / 4 row is padded by 64 bytes, which spreads both the writes (a wavefront writes whole rows
// of an x-fast operand, 16 x of four rows of a k-fast one) and the reads (16 x of eight rows) over all
// banks.  An x-fast fetch brings four consecutive x, which go to four positions a quarter of the
// tile apart: so the writes of neighbouring lanes are neighbours, and the four blocks of 16
// positions that a wavefront takes give a lane four consecutive rows of the result, stored as 16
// bytes without a further pass through LDS.
//
// What bounds it: a 16 x 16 x 32 instruction holds its matrix core for 16 cycles and the vector
// unit for 8, so two vector instructions per matrix instruction are free (measured; each further
// one costs its 4 cycles).  The cut takes 13 per two values, i.e. 1.6 per matrix instruction on
// the 256 x 128 tile and 2.2 on the 128 x 128 one.  Sustained, the chip's power decides: 100%
// matrix work runs at 1.87 GHz.
#pragma once
#include "gemm_core.h"

#ifdef __HIPCC__
typedef __bf16 mnv_bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 mnv_bf8 __attribute__((ext_vector_type(8)));
typedef unsigned mnv_u2 __attribute__((ext_vector_type(2)));
typedef unsigned mnv_u4 __attribute__((ext_vector_type(4)));

#define MNV_SPLIT_SCALE 65536.f                  // 2^16, of either operand
#define MNV_SPLIT_UNSCALE 2.3283064365386963e-10f  // 2^-32, of the product

// BUFS 2: the next step's planes are written while this one's are multiplied (one barrier per
// step; the workgroup has the CU to itself).  BUFS 1: one set of planes and two barriers, and two
// workgroups per CU, each multiplying while the other cuts.
// BNU: columns of the tile that are multiplied (see MnvGemmTile).
template <int BM_, int BN_, int WGM_, int WGN_, int BUFS_, int BNU_ = BN_>
struct MnvSplitTile {
  static constexpr bool SPLIT = true;
  static constexpr int BM = BM_, BN = BN_, BNU = BNU_, BK = 16, WGM = WGM_, WGN = WGN_, BUFS = BUFS_;
  static constexpr int NT = MNV_WAVE * WGM * WGN, NG = NT / 2;  // NG: threads that fetch one slab
  static constexpr int WM = BM / WGM, WN = BNU / WGN, TM = WM / 16, TN = WN / 16;
  static constexpr int pitch(int bx) { return bx * 8 + 64; }  // bytes of a k / 4 row
  static constexpr int plane(int bx) { return 8 * pitch(bx); }
  static constexpr int A_BYTES = 3 * plane(BM), B_BYTES = 3 * plane(BN), BUF_BYTES = A_BYTES + B_BYTES;
  static constexpr size_t lds_bytes(bool, bool) { return (size_t)BUFS * BUF_BYTES; }
  static constexpr int MIN_WAVES = NT / 256 * (3 - BUFS);  // per SIMD
  // One workgroup per CU as the gathers of the convolutions run on it, two on 96 and 128 columns (see mnv_tail_plan).
  static constexpr MnvTailCost TAIL = BUFS == 2 ? MnvTailCost{0.8, 3.0} : BNU == 96 ? MnvTailCost{1.1, 1.5} : MnvTailCost{0.72, 1.5};
  static_assert(TM == 4 && WM % 16 == 0 && WN % 16 == 0 && BM % 64 == 0 && BN % 32 == 0, "four blocks of rows per wavefront");
};

// two values (consecutive k of one x) as three pairs of bf16, the largest first
__device__ __forceinline__ unsigned mnv_pack_bf16(float x, float y) {
  const mnv_bf2 t = {(__bf16)x, (__bf16)y};
  unsigned u = __builtin_bit_cast(unsigned, t);
  asm("" : "+v"(u));  // one conversion of both: left alone, the compiler converts each again for its half
  return u;
}
__device__ __forceinline__ void mnv_split_pair(float x, float y, float scale, unsigned (&p)[3]) {
  x *= scale;
  y *= scale;
  p[0] = mnv_pack_bf16(x, y);
  x -= __builtin_bit_cast(float, p[0] << 16);
  y -= __builtin_bit_cast(float, p[0] & 0xffff0000u);
  p[1] = mnv_pack_bf16(x, y);
  x -= __builtin_bit_cast(float, p[1] << 16);
  y -= __builtin_bit_cast(float, p[1] & 0xffff0000u);
  p[2] = mnv_pack_bf16(x, y);
}

// Where the values of an operand tile (BX x 16, fetched by NG threads) are, in the fetches and in LDS.
template <int BX, int NG, bool KFAST, int XPK>
struct MnvSplitMap {
  static constexpr int XP = KFAST ? XPK : 4, QX = BX / XP;  // neighbouring x lie QX positions apart
  // vectors per thread: x-fast, V consecutive k of the same four x; k-fast, four k of V different x
  static constexpr int V = BX * 16 / (4 * NG);
  static constexpr int PIECES = KFAST ? V : 4;
  static_assert(BX * 16 % (4 * NG) == 0 && (KFAST ? V >= 1 : V == 2 || V == 4), "tile/thread mismatch");
  __device__ static int x(int g, int p) {
    if (!KFAST) return g % QX * 4;
    const int pos = g / 4 + NG / 4 * p;
    return XP * (pos % QX) + pos / QX;
  }
  __device__ static int k(int g, int p) { return KFAST ? g % 4 * 4 : g / QX * V + p; }
  // Block q of 16 positions, counted so that XP consecutive blocks hold neighbouring x: row r of
  // it is x = block_x(q) + XP r.
  __device__ static int block_pos(int q) { return q % XP * QX + q / XP * 16; }
  __device__ static int block_x(int q) { return q / XP * 16 * XP + q % XP; }
  // cuts the vectors v of slab `sub` of the step, pieces [from, to), into the planes
  __device__ static void stash(char* planes, int g, int sub, float scale, const float (&v)[V][4], int from, int to) {
    constexpr int PITCH = BX * 8 + 64, PLANE = 8 * PITCH;
    if constexpr (KFAST) {
      char* at = planes + (sub * 4 + g % 4) * PITCH + g / 4 * 8;
#pragma unroll
      for (int p = from; p < to; ++p) {
        unsigned lo[3], hi[3];
        mnv_split_pair(v[p][0], v[p][1], scale, lo);
        mnv_split_pair(v[p][2], v[p][3], scale, hi);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
          *reinterpret_cast<mnv_u2*>(at + pl * PLANE + p * (NG / 4) * 8) = mnv_u2{lo[pl], hi[pl]};
      }
    } else {
      const int kb = g / QX;
      char* at = planes + (sub * 4 + kb * V / 4) * PITCH + g % QX * 8 + (V == 2 ? (kb & 1) * 4 : 0);
#pragma unroll
      for (int i = from; i < to; ++i) {
        unsigned lo[3], hi[3];
        mnv_split_pair(v[0][i], v[1][i], scale, lo);
        if constexpr (V == 4) mnv_split_pair(v[2][i], v[3][i], scale, hi);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) {
          if constexpr (V == 4) *reinterpret_cast<mnv_u2*>(at + pl * PLANE + i * QX * 8) = mnv_u2{lo[pl], hi[pl]};
          else *reinterpret_cast<unsigned*>(at + pl * PLANE + i * QX * 8) = lo[pl];
        }
      }
    }
  }
};

// four consecutive rows of one column; m < M, n < N
template <class P>
__device__ __forceinline__ void mnv_split_store4(const P& prob, int m, int n, const float (&x)[4]) {
  if constexpr (MnvCStore4<P>::value) {
    prob.c_store4(m, n, x);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (m + q < prob.M) prob.c_store(m + q, n, x[q]);
  }
}

// A wavefront's block again, with the fp32 instruction: for sums that are not all finite.  Every
// lane fetches its own rows through the policy, no LDS and no barrier.  Instruction t of a slab
// takes k = 4 (lane / 16) + t of both operands.
template <class T, class P, class MapA, class MapB, class Acc>
__device__ __forceinline__ void mnv_split_redo(const P& prob, const typename P::Res& res, int m0, int n0, int wm, int wn,
                                               int lane, int slab_begin, int slab_end, Acc (&acc)[T::TM][T::TN]) {
  const int lr = lane % 16, lq = lane / 16;
#pragma unroll
  for (int i = 0; i < T::TM; ++i)
#pragma unroll
    for (int j = 0; j < T::TN; ++j) acc[i][j] = Acc{0.f, 0.f, 0.f, 0.f};
  auto pick = [](const float (&v)[4], int e) { return e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3]; };
#pragma unroll 1
  for (int slab = slab_begin; slab < slab_end; ++slab) {
    const int period = slab / prob.spp, s = slab - period * prob.spp;
    float av[T::TM][4], bv[T::TN][4];
#pragma unroll
    for (int i = 0; i < T::TM; ++i) {
      const int x = MapA::block_x(wm * T::TM + i) + MapA::XP * lr, m = m0 + (P::A_KFAST ? x : x / 4 * 4);
      typename P::AState st;
      unsigned off[P::A_NOFF];
      prob.a_init(res, st, m);
#pragma unroll
      for (int t = 0; t < (P::A_KFAST ? 1 : 4); ++t) {
        const int kl = 4 * lq + t;
        float v[4];
        prob.a_period(st, off, m, kl, period);
        prob.a_load(res, st, off, period, s, kl, v);
        if constexpr (MnvAStashFix<P>::value) prob.a_stash_fix(period, s, kl, v);
        if (P::A_KFAST) {
#pragma unroll
          for (int q = 0; q < 4; ++q) av[i][q] = v[q];
        } else {
          av[i][t] = pick(v, x % 4);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < T::TN; ++j) {
      const int x = MapB::block_x(wn * T::TN + j) + MapB::XP * lr, n = n0 + (P::B_KFAST ? x : x / 4 * 4);
      typename P::BState st;
      unsigned off[P::B_NOFF];
      prob.b_init(res, st, n);
#pragma unroll
      for (int t = 0; t < (P::B_KFAST ? 1 : 4); ++t) {
        const int kl = 4 * lq + t;
        float v[4];
        prob.b_period(st, off, n, kl, period);
        prob.b_load(res, st, off, period, s, kl, v);
        if constexpr (MnvBStashFix<P>::value) prob.b_stash_fix(period, s, kl, v);
        if (P::B_KFAST) {
#pragma unroll
          for (int q = 0; q < 4; ++q) bv[j][q] = v[q];
        } else {
          bv[j][t] = pick(v, x % 4);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < T::TM; ++i)
#pragma unroll
        for (int j = 0; j < T::TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j][t], av[i][t], acc[i][j], 0, 0, 0);
  }
}

// Arguments, k ranges, cut tails and stream-k plans as in mnv_gemm_kernel.  Partial tiles are kept
// in register order as there, a 16-byte group being four consecutive rows of one column here: group
// j 4 + r of a thread is column r of its lane's four in block column j.
template <class T, class P, bool SK = false>
__global__ __launch_bounds__(T::NT, T::MIN_WAVES) void mnv_gemm_split_kernel(P prob, int tiles_m, int tiles_n,
                                                                             int slabs_per_split,
                                                                             float* __restrict__ partial,
                                                                             int tail_begin, int tail_z) {
  static_assert(!MnvALaneK<P>::value, "a fetch of one k per lane has no pairs to cut");
  extern __shared__ __align__(16) char mnv_split_lds[];
  typedef MnvSplitMap<T::BM, T::NG, P::A_KFAST, 4> MapA;
  typedef MnvSplitMap<T::BN, T::NG, P::B_KFAST, 1> MapB;
  static_assert(T::BNU == T::BN || P::B_KFAST, "only neighbouring positions can be left out");
  const int tid = threadIdx.x, g = tid % T::NG;
  const int wave = __builtin_amdgcn_readfirstlane(tid / MNV_WAVE), lane = tid % MNV_WAVE;
  const int sub = wave / (T::NG / MNV_WAVE);
  const int wm = wave % T::WGM, wn = wave / T::WGM, lr = lane % 16, lq = lane / 16;
  const int tiles = tiles_m * tiles_n;

  long long sk_u = 0, sk_end = 0;
  int sk_p = 0, sk_aligned = 0, sk_rest = 0;
  if constexpr (SK) {
    const int aligned = tiles * tail_begin, rem = (int)gridDim.x - aligned;
    sk_p = mnv_tile_remap((int)blockIdx.x, (int)gridDim.x);
    sk_aligned = sk_p < aligned;
    sk_rest = prob.total_slabs - tail_begin * slabs_per_split;
    if (!sk_aligned) {
      const long long units = (long long)sk_rest * tiles;
      sk_u = units * (sk_p - aligned) / rem;
      sk_end = units * (sk_p - aligned + 1) / rem;
      if (sk_u >= sk_end) return;
    }
  }
  for (;;) {  // SK: one pass per segment; otherwise a single pass that ends in a return
    int vb = blockIdx.x, tail_part = -1, tile_m, tile_n, slab_begin, slab_end;
    if constexpr (SK) {
      if (sk_aligned) {
        const int z = sk_p / tiles;
        vb = sk_p - z * tiles;
        if ((int)gridDim.x == tiles * tail_begin) {
          slab_begin = (int)((long long)prob.total_slabs * z / tail_begin);
          slab_end = (int)((long long)prob.total_slabs * (z + 1) / tail_begin);
        } else {
          slab_begin = z * slabs_per_split;
          slab_end = slab_begin + slabs_per_split;
        }
      } else {
        vb = (int)(sk_u / sk_rest);
        slab_begin = prob.total_slabs - sk_rest + (int)(sk_u - (long long)vb * sk_rest);
        const long long left = sk_end - sk_u;
        slab_end = left < prob.total_slabs - slab_begin ? slab_begin + (int)left : prob.total_slabs;
      }
      tile_m = vb % tiles_m;
      tile_n = vb / tiles_m;
    } else {
      if (tail_z > 1 && vb >= tail_begin) {
        const int i = vb - tail_begin, tl = i / tail_z;
        tail_part = i - tl * tail_z;
        vb = tail_begin + tl;
      }
      mnv_tile_coords(prob, vb, T::BM, tiles_m, tiles_n, tile_m, tile_n);
      const int total_slabs = mnv_tile_slabs(prob, tile_m * T::BM, slabs_per_split);
      int per = slabs_per_split, begin = blockIdx.z * per;
      if (tail_part >= 0) {
        per = (total_slabs + tail_z - 1) / tail_z;
        begin = tail_part * per;
      }
      slab_begin = begin < total_slabs ? begin : total_slabs;
      slab_end = begin + per < total_slabs ? begin + per : total_slabs;
    }
    const int m0 = tile_m * T::BM, n0 = tile_n * T::BNU;

    typename P::Res res;
    prob.make_res(res);
    prob.block_init(res, reinterpret_cast<float*>(mnv_split_lds + T::BUFS * T::BUF_BYTES), m0, n0);
    typename P::AState ast[MapA::V];
    typename P::BState bst[MapB::V];
    unsigned aoff[MapA::V][P::A_NOFF], boff[MapB::V][P::B_NOFF];
#pragma unroll
    for (int p = 0; p < MapA::V; ++p) prob.a_init(res, ast[p], m0 + MapA::x(g, p));
#pragma unroll
    for (int p = 0; p < MapB::V; ++p) prob.b_init(res, bst[p], n0 + MapB::x(g, p));
    float ra[MapA::V][4], rb[MapB::V][4];
    // The wavefront's slab, its period and place in it.  Past the end of the k range the last
    // fetch is repeated and its values are multiplied by 0 (a NaN from that goes the way of
    // every sum that is not finite, and an operand that gives one is not finite).
    int slab = slab_begin + sub, held_period = 0, held_s = 0;
    float held_scale = 0.f;
    bool live = slab < slab_end;
    if (!live) slab = slab_begin;
    int period = slab / prob.spp, s = slab - period * prob.spp;
    auto new_period = [&]() {
#pragma unroll
      for (int p = 0; p < MapA::V; ++p) prob.a_period(ast[p], aoff[p], m0 + MapA::x(g, p), MapA::k(g, p), period);
#pragma unroll
      for (int p = 0; p < MapB::V; ++p) prob.b_period(bst[p], boff[p], n0 + MapB::x(g, p), MapB::k(g, p), period);
    };
    auto advance = [&]() {
      slab += 2;
      live = slab < slab_end;
      if (live) {
        s += 2;
        if (s >= prob.spp) {
          do {
            s -= prob.spp;
            ++period;
          } while (s >= prob.spp);
          new_period();
        }
      }
    };
    auto fetch_a = [&]() {
#pragma unroll
      for (int p = 0; p < MapA::V; ++p) prob.a_load(res, ast[p], aoff[p], period, s, MapA::k(g, p), ra[p]);
    };
    auto fetch_b = [&]() {
#pragma unroll
      for (int p = 0; p < MapB::V; ++p) prob.b_load(res, bst[p], boff[p], period, s, MapB::k(g, p), rb[p]);
      held_period = period;
      held_s = s;
      held_scale = live ? MNV_SPLIT_SCALE : 0.f;
    };
    auto stash_a = [&](int at, int from, int to) {
      if constexpr (MnvAStashFix<P>::value) {
        static_assert(P::A_KFAST, "pieces are vectors");
#pragma unroll
        for (int p = from; p < to; ++p) prob.a_stash_fix(held_period, held_s, MapA::k(g, p), ra[p]);
      }
      MapA::stash(mnv_split_lds + at, g, sub, held_scale, ra, from, to);
    };
    auto stash_b = [&](int at) {
      if constexpr (MnvBStashFix<P>::value) {
#pragma unroll
        for (int p = 0; p < MapB::V; ++p) prob.b_stash_fix(held_period, held_s, MapB::k(g, p), rb[p]);
      }
      MapB::stash(mnv_split_lds + at + T::A_BYTES, g, sub, held_scale, rb, 0, MapB::PIECES);
    };
    typedef float Acc __attribute__((ext_vector_type(4)));
    Acc acc[T::TM][T::TN], low[T::TM][T::TN];
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
      for (int j = 0; j < T::TN; ++j) acc[i][j] = low[i][j] = Acc{0.f, 0.f, 0.f, 0.f};

    __syncthreads();  // block_init may have written LDS
    if (slab_begin < slab_end) {
      new_period();
      fetch_a();
      fetch_b();
      stash_a(0, 0, MapA::PIECES);
      stash_b(0);
      advance();
      fetch_a();
      fetch_b();
    }
    __syncthreads();
    constexpr int PA = T::pitch(T::BM), PB = T::pitch(T::BN);
    // The eight k of a lane as two 8-byte reads.  volatile keeps the compiler from pairing them with
    // those of the neighbouring block, which it would take apart with moves.
    auto frag = [&](const char* at, int pitch) -> mnv_bf8 {
      typedef const volatile __attribute__((address_space(3))) mnv_u2* Lds;
      const mnv_u2 lo = *(Lds)at, hi = *(Lds)(at + pitch);
      return __builtin_bit_cast(mnv_bf8, mnv_u4{lo.x, lo.y, hi.x, hi.y});
    };
    const int steps = (slab_end - slab_begin + 1) / 2;
#pragma unroll 1
    for (int it = 0, at = 0; it < steps; ++it) {
      const int next = T::BUFS == 1 ? 0 : T::BUF_BYTES - at;
      const char* a = mnv_split_lds + at + MapA::block_pos(wm * T::TM) * 8 + 2 * lq * PA + lr * 8;
      const char* bb = mnv_split_lds + at + MapB::block_pos(wn * T::TN) * 8 + T::A_BYTES + 2 * lq * PB + lr * 8;
      mnv_bf8 bf[T::TN][3];
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
#pragma unroll
        for (int j = 0; j < T::TN; ++j) bf[j][pl] = frag(bb + MapB::block_pos(j) * 8 + pl * 8 * PB, PB);
#pragma unroll
      for (int i = 0; i < T::TM; ++i) {
        mnv_bf8 af[3];
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) af[pl] = frag(a + MapA::block_pos(i) * 8 + pl * 8 * PA, PA);
        if (T::BUFS == 2 && i == 2) advance();
        auto multiply = [&](int pa, int pb, Acc(&to)[T::TN]) {
#pragma unroll
          for (int j = 0; j < T::TN; ++j) to[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j][pb], af[pa], to[j], 0, 0, 0);
        };
        multiply(2, 0, low[i]);
        multiply(0, 0, acc[i]);
        multiply(1, 1, low[i]);
        multiply(0, 2, low[i]);
        multiply(1, 0, low[i]);
        multiply(0, 1, low[i]);
        // The cut of the next step and the loads of the one after it, in parts between the
        // multiplies; the barrier keeps the scheduler from gathering them in one place.
        if (T::BUFS == 2) {
          if (i == 0) stash_a(next, 0, MapA::PIECES / 2);
          if (i == 1) stash_a(next, MapA::PIECES / 2, MapA::PIECES);
          if (i == 2) {
            stash_b(next);
            fetch_a();
          }
          if (i == 3) fetch_b();
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (T::BUFS == 1 && it + 1 < steps) {
        __syncthreads();
        stash_a(0, 0, MapA::PIECES);
        stash_b(0);
        advance();
        fetch_a();
        fetch_b();
      }
      at = next;
      __syncthreads();
    }

    // Register r of lane (lr, lq) holds row lr and column 4 lq + r of its 16 x 16 block.
    float finite = 0.f;
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
      for (int j = 0; j < T::TN; ++j) {
        acc[i][j] = (acc[i][j] + low[i][j]) * MNV_SPLIT_UNSCALE;
#pragma unroll
        for (int r = 0; r < 4; ++r) finite = __builtin_fmaf(acc[i][j][r], 0.f, finite);
      }
    if (__any(!(finite == 0.f)))
      mnv_split_redo<T, P, MapA, MapB>(prob, res, m0, n0, wm, wn, lane, slab_begin, slab_end, acc);

    if (SK || tail_part >= 0) {  // the whole tile, in register order, into its slot
      int at = tid * 4;
      asm volatile("" : "+v"(at));  // not computed ahead of the main loop and held through it
      const size_t slot = SK ? (size_t)(sk_aligned ? sk_p : sk_p + vb) : (size_t)(vb - tail_begin) * tail_z + tail_part;
      float* pt = partial + slot * (T::BM * T::BNU) + at;
#pragma unroll
      for (int j = 0; j < T::TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *reinterpret_cast<mnv_f4*>(pt + (j * 4 + r) * (T::NT * 4)) =
              mnv_f4{acc[0][j][r], acc[1][j][r], acc[2][j][r], acc[3][j][r]};
      if (!SK || sk_aligned) return;
      sk_u += slab_end - slab_begin;
      if (sk_u >= sk_end) return;
      __syncthreads();  // mnv_split_redo may read the policy's LDS
      continue;
    }
    const bool split = gridDim.z > 1;
    float* part = split ? partial + (size_t)blockIdx.z * prob.M * prob.N : nullptr;
    const int m = m0 + MapA::block_x(wm * T::TM) + MapA::XP * lr;
    if (m >= prob.M) return;
#pragma unroll
    for (int j = 0; j < T::TN; ++j) {
      const int nj = n0 + MapB::block_x(wn * T::TN + j) + MapB::XP * 4 * lq;
      if constexpr (MnvCPreload<P>::value) {
        if (!split && prob.c_preload_on()) {
          float pre[4][4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              pre[r][q] = nj + MapB::XP * r < prob.N && m + q < prob.M ? prob.c_preload(m + q, nj + MapB::XP * r) : 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (nj + MapB::XP * r < prob.N && m + q < prob.M) prob.c_store_with(m + q, nj + MapB::XP * r, acc[q][j][r], pre[r][q]);
          continue;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = nj + MapB::XP * r;
        if (n >= prob.N) continue;
        const float x[4] = {acc[0][j][r], acc[1][j][r], acc[2][j][r], acc[3][j][r]};
        if (!split) {
          mnv_split_store4(prob, m, n, x);
        } else if (m + 3 < prob.M) {
          *reinterpret_cast<mnv_f4u*>(part + (size_t)n * prob.M + m) = mnv_f4u{x[0], x[1], x[2], x[3]};
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (m + q < prob.M) part[(size_t)n * prob.M + m + q] = x[q];
        }
      }
    }
    return;
  }
}
#endif  // __HIPCC__
