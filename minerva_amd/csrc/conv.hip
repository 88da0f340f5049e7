// Convolution forward, backward-data and backward-filter as implicit GEMMs on the matrix cores:
// with the fp32 instruction (gemm_core.h) or, where that is the faster one, in bf16 parts
// (gemm_split.h).  Semantics: cuDNN v2 CUDNN_CONVOLUTION (flipped filter),
// zero padding, NCHW / KCRS bytes, as selected by the reference at
// minerva/op/impl/cuda/cuda_perform.cu:227-318:
//   top[n,k,i,j] = bias[k] + sum_{c,r,s} bottom[n,c,i*sv-ph+r,j*sh-pw+s] * filter[k,c,R-1-r,S-1-s]
// With r' = R-1-r, s' = S-1-s the filter is read in its natural order, so it is a plain
// column-major {C*R*S, K} matrix, and the flip moves into the im2col gather.
//
//   forward        : C[(n,i,j), k]      = sum_{(c,r',s')}  im2col(bottom) * filter
//   backward data  : C[(n,y,x), c]      = sum_{(k,r',s')}  gather(top_diff) * filter^T-gather
//   backward filter: C[(c,r',s'), k]    = sum_{(n,i,j)}    gather(bottom) * top_diff   (k range split)
// In every case the GEMM "m" dimension is the one that is contiguous in the output
// tensor, so result stores are coalesced, and no im2col buffer exists in HBM.
// Roofline: 2*N*Ho*Wo*K*C*R*S algorithmic flops per pass, at 157.3 TFLOP/s with the fp32 instruction and 419.4
// in parts (six bf16 products of 2516.6).

#include "gemm_split.h"
#include "winograd.h"

namespace {

struct ConvGeom {
  int N, C, K, H, W, Ho, Wo, R, S, ph, pw, sv, sh;
  int HW, HoWo, RS, CRS;
  MnvFastDiv d_RS, d_S, d_HoWo, d_Wo, d_HW, d_W, d_sv, d_sh;
};

#define MNV_FAR (-20000)  // row/col origin that fails every bounds test

__device__ __forceinline__ int pack_yx(int y, int x) { return (y << 16) | (x & 0xffff); }
__device__ __forceinline__ int unpack_y(int p) { return p >> 16; }
__device__ __forceinline__ int unpack_x(int p) { return (int)(short)(p & 0xffff); }

// Every policy comes in two addressing flavours (see the contract in gemm_core.h):
//   FAST   : the reduction index is ordered (filter tap, channel) and a period is one tap,
//            so the im2col offsets and their bounds tests are computed once per tap and a
//            slab of 16 channels only advances a uniform scalar offset.  Takes the channels
//            of the reduction 16 at a time (and unit stride for the data gradient); PAD: their
//            count is no multiple of 16, the permuted filter is padded with zeros to one and
//            the missing channels of the last slab of a tap read as 0 too (not as the next
//            image, whose infinities the zeros would turn into NaN).
//   generic: the reduction index is the flat (channel, tap) order, one period per slab.
// The two orders only differ in the order the products are summed.

// ------------------------------------------------------------------ forward
template <bool FAST, bool PAD = false>
struct ConvFwd {
  static constexpr bool A_KFAST = false, B_KFAST = true;
  static constexpr int A_NOFF = 4, B_NOFF = FAST ? 1 : 4;
  const float* __restrict__ bottom;
  const float* __restrict__ filter;
  const float* __restrict__ bias;
  float* __restrict__ top;
  ConvGeom g;
  int M, N, K, total_slabs, spp;  // GEMM extents: N*Ho*Wo, Kout, C*R*S
  int relu;                       // fused epilogue: top = max(conv + bias, 0)
  struct Res {
    mnv_rsrc a, b;
  };
  struct AState {
    int off[4], yx[4];
  };
  struct BState {};
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(bottom, (unsigned)(g.N * g.C * g.HW) * 4u);
    r.b = mnv_make_rsrc(filter, (unsigned)(FAST ? N * g.RS * spp * 16 : g.K * g.CRS) * 4u);
  }
  __device__ void a_init(const Res& res, AState& st, int m) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int mm = m + q;
      int img = mnv_fastdiv(mm, g.d_HoWo);
      int pos = mm - img * g.HoWo;
      int i = mnv_fastdiv(pos, g.d_Wo);
      int j = pos - i * g.Wo;
      int y0 = i * g.sv - g.ph, x0 = j * g.sh - g.pw;
      st.off[q] = img * g.C * g.HW + y0 * g.W + x0;
      st.yx[q] = mm < M ? pack_yx(y0, x0) : pack_yx(MNV_FAR, MNV_FAR);
    }
  }
  __device__ void b_init(const Res&, BState&, int) const {}
  __device__ void a_period(const AState& st, unsigned (&off)[4], int, int kl, int period) const {
    int c, rs;
    bool kok = true;
    if (FAST) {  // period = tap, kl = channel within the slab
      rs = period;
      c = kl;
    } else {  // period = slab, flat k = (c, r', s')
      int k = period * 16 + kl;
      kok = k < K;
      c = mnv_fastdiv(k, g.d_RS);
      rs = k - c * g.RS;
    }
    int rp = mnv_fastdiv(rs, g.d_S);
    int sp = rs - rp * g.S;
    int r = g.R - 1 - rp, s = g.S - 1 - sp;  // flipped tap
    int koff = c * g.HW + r * g.W + s;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int y = unpack_y(st.yx[q]) + r, x = unpack_x(st.yx[q]) + s;
      bool ok = kok & ((unsigned)y < (unsigned)g.H) & ((unsigned)x < (unsigned)g.W);
      off[q] = ok ? (unsigned)(st.off[q] + koff) * 4u : MNV_OOB;
    }
  }
  __device__ void a_load(const Res& r, const AState&, const unsigned (&off)[4], int, int s, int kl,
                         float (&v)[4]) const {
    const unsigned slab = FAST ? (unsigned)s * 16u * (unsigned)g.HW * 4u : 0u;
    if (PAD) {
      const bool ok = s * 16 + kl < g.C;
      const unsigned in[4] = {ok ? off[0] : MNV_OOB, ok ? off[1] : MNV_OOB, ok ? off[2] : MNV_OOB, ok ? off[3] : MNV_OOB};
      mnv_fetch_vec<4>(r.a, in, slab, v);
    } else {
      mnv_fetch_vec<4>(r.a, off, slab, v);
    }
  }
  __device__ int channels() const { return g.C; }
  __device__ int channel_floats() const { return g.HW; }
  size_t extra_lds_bytes() const { return 0; }
  __device__ void block_init(Res&, float*, int, int) const {}
  // generic: `filter` is the caller's tensor [n][c][r'][s'], element (k, n) at n*CRS + k.
  // FAST: `filter` is the permuted copy [n][r's'][c, padded to 16], so the 4 channels of a vector are
  // one 16-byte load and consecutive slabs are consecutive memory.
  __device__ void b_period(const BState&, unsigned (&off)[B_NOFF], int n, int kl,
                           int period) const {
    if (FAST) {
      off[0] = (n < N) ? (unsigned)((n * g.RS + period) * spp * 16 + kl) * 4u : MNV_OOB;
    } else {
#pragma unroll
      for (int q = 0; q < B_NOFF; ++q) {
        int k = period * 16 + kl + q;
        off[q] = ((n < N) & (k < K)) ? (unsigned)(n * K + k) * 4u : MNV_OOB;
      }
    }
  }
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[B_NOFF], int, int s,
                         int, float (&v)[4]) const {
    mnv_fetch_vec<B_NOFF>(r.b, off, FAST ? (unsigned)s * 64u : 0u, v);
  }
  // The fused ReLU is the selection mnv_relu_fwd makes on the stored value, so the result has
  // the bits of the two-operator sequence.
  __device__ void c_store(int m, int n, float x) const {
    int img = mnv_fastdiv(m, g.d_HoWo);
    int pos = m - img * g.HoWo;
    float v = x + bias[n];
    if (relu) v = v > 0.f ? v : 0.f;
    top[((size_t)img * N + n) * g.HoWo + pos] = v;
  }
  // four consecutive positions of one channel: one 16-byte store (4-byte aligned) unless the
  // four straddle two images or the end of the batch
  static constexpr bool C_STORE4 = true;
  __device__ void c_store4(int m, int n, const float (&x)[4]) const {
    int img = mnv_fastdiv(m, g.d_HoWo);
    int pos = m - img * g.HoWo;
    if (m + 3 < M && pos + 3 < g.HoWo) {
      const float b = bias[n];
      mnv_f4u v = {x[0] + b, x[1] + b, x[2] + b, x[3] + b};
      if (relu) {
        v.x = v.x > 0.f ? v.x : 0.f; v.y = v.y > 0.f ? v.y : 0.f;
        v.z = v.z > 0.f ? v.z : 0.f; v.w = v.w > 0.f ? v.w : 0.f;
      }
      *reinterpret_cast<mnv_f4u*>(top + ((size_t)img * N + n) * g.HoWo + pos) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (m + q < M) c_store(m + q, n, x[q]);
    }
  }
};

// Forward without padding (ph == pw == 0, any channel count and stride).  Every tap of
// every output position is a real pixel, so the pixel offset is base(position) + koff(k)
// with koff(k) = ((c*H + R-1-r')*W + S-1-s')*4 for the flat reduction index k = (c, r', s').
// koff is tabulated in LDS once per workgroup; a slab then costs one 16-byte LDS read and
// four adds per vector, and nothing is decomposed or bounds-tested in the main loop.  The
// filter needs no copy: in this order it already is the column-major K x Kout operand.
// Period 0 holds the full slabs, period 1 the last, partial one (masked filter loads).
// A vector is four consecutive k at ONE output position (k-fast): its four loads are 4-byte
// gathers either way, but with four lanes per position a load instruction touches about 20
// cache lines (16 positions, the taps of a vector a few floats apart) where four
// consecutive positions per lane touched 64 at a stride of four pixels -- and conv1
// (stride 4, C = 3) was bound by those L1 look-ups, not by the matrix pipe.
struct ConvFwdNP {
  static constexpr bool A_KFAST = true, B_KFAST = true;
  static constexpr int A_NOFF = 1, B_NOFF = 4;
  const float* __restrict__ bottom;
  const float* __restrict__ filter;
  const float* __restrict__ bias;
  float* __restrict__ top;
  ConvGeom g;
  int M, N, K, total_slabs, spp;  // GEMM extents: N*Ho*Wo, Kout, C*R*S
  int relu;                       // fused epilogue: top = max(conv + bias, 0)
  struct Res {
    mnv_rsrc a, b;
    const unsigned* tab;  // LDS: [total_slabs*16] byte offsets, MNV_OOB past K
  };
  struct AState {};
  struct BState {};
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(bottom, (unsigned)(g.N * g.C * g.HW) * 4u);
    r.b = mnv_make_rsrc(filter, (unsigned)(g.K * g.CRS) * 4u);
    r.tab = nullptr;
  }
  size_t extra_lds_bytes() const { return (size_t)total_slabs * 16 * sizeof(unsigned); }
  __device__ void block_init(Res& r, float* extra, int, int) const {
    unsigned* tab = reinterpret_cast<unsigned*>(extra);
    r.tab = tab;
    for (int k = threadIdx.x; k < total_slabs * 16; k += blockDim.x) {
      int c = mnv_fastdiv(k, g.d_RS);
      int rs = k - c * g.RS;
      int rp = mnv_fastdiv(rs, g.d_S), sp = rs - rp * g.S;
      tab[k] = k < K ? (unsigned)(c * g.HW + (g.R - 1 - rp) * g.W + (g.S - 1 - sp)) * 4u : MNV_OOB;
    }
  }
  __device__ void a_init(const Res&, AState&, int) const {}
  __device__ void b_init(const Res&, BState&, int) const {}
  // rows past M are never stored, so they may read any valid pixel
  __device__ void a_period(const AState&, unsigned (&off)[1], int m, int, int) const {
    int mm = m < M ? m : 0;
    int img = mnv_fastdiv(mm, g.d_HoWo);
    int pos = mm - img * g.HoWo;
    int i = mnv_fastdiv(pos, g.d_Wo);
    int j = pos - i * g.Wo;
    off[0] = (unsigned)(img * g.C * g.HW + i * g.sv * g.W + j * g.sh) * 4u;
  }
  // an entry past K is MNV_OOB, and MNV_OOB plus any pixel offset is still out of range
  __device__ void a_load(const Res& r, const AState&, const unsigned (&off)[1], int period, int s,
                         int kl, float (&v)[4]) const {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const u4 t = *reinterpret_cast<const u4*>(
        __builtin_assume_aligned(r.tab + (period * spp + s) * 16 + kl, 16));
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = __builtin_bit_cast(float,
                                __builtin_amdgcn_raw_buffer_load_b32(r.a, (int)(off[0] + t[q]), 0, 0));
  }
  // filter element (k, n) at n*K + k: four consecutive k are one 16-byte load (4-byte
  // aligned is enough for a buffer load)
  __device__ void b_period(const BState&, unsigned (&off)[4], int n, int kl, int period) const {
    int k = period * spp * 16 + kl;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      off[q] = ((n < N) & (k + q < K)) ? (unsigned)(n * K + k + q) * 4u : MNV_OOB;
  }
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[4], int period, int s,
                         int, float (&v)[4]) const {
    if (period == 0 && spp * 16 <= K) {  // uniform: a full slab
      const unsigned one[1] = {off[0]};
      mnv_fetch_vec<1>(r.b, one, (unsigned)s * 64u, v);
    } else {
      mnv_fetch_vec<4>(r.b, off, (unsigned)s * 64u, v);
    }
  }
  __device__ void c_store(int m, int n, float x) const {
    int img = mnv_fastdiv(m, g.d_HoWo);
    int pos = m - img * g.HoWo;
    float v = x + bias[n];
    if (relu) v = v > 0.f ? v : 0.f;
    top[((size_t)img * N + n) * g.HoWo + pos] = v;
  }
  // four consecutive positions of one channel: one 16-byte store (4-byte aligned) unless the
  // four straddle two images or the end of the batch
  static constexpr bool C_STORE4 = true;
  __device__ void c_store4(int m, int n, const float (&x)[4]) const {
    int img = mnv_fastdiv(m, g.d_HoWo);
    int pos = m - img * g.HoWo;
    if (m + 3 < M && pos + 3 < g.HoWo) {
      const float b = bias[n];
      mnv_f4u v = {x[0] + b, x[1] + b, x[2] + b, x[3] + b};
      if (relu) {
        v.x = v.x > 0.f ? v.x : 0.f; v.y = v.y > 0.f ? v.y : 0.f;
        v.z = v.z > 0.f ? v.z : 0.f; v.w = v.w > 0.f ? v.w : 0.f;
      }
      *reinterpret_cast<mnv_f4u*>(top + ((size_t)img * N + n) * g.HoWo + pos) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (m + q < M) c_store(m + q, n, x[q]);
    }
  }
};

// The same with the filter's rows cut into groups of four taps, for filters whose rows are a multiple
// of four taps long or one short of it (11: 12 slots for 11 taps): a vector is then four neighbouring
// pixels and four neighbouring filter values, one 16-byte load (4-byte aligned) each, where the
// flat order's vectors straddle filter rows and take a 4-byte load per pixel.  The order of the
// slots of a group is that of the pixels, against that of the taps.  A row's last group ends with the
// row as well and so begins with a tap that the group before it has: its slot 3 reads as 0 in both operands.
// The table holds, for every group, the byte offsets of its pixels and its filter values.  3 -> 96 channels under 11 x 11
// at stride 4 on 256 x 227 x
// 227: 555 us with the fp32 instruction, 537 in parts in the flat order, 432 so.
struct ConvFwdRows : ConvFwdNP {
  static constexpr int B_NOFF = 1;
  int groups, per_row;  // C * R * per_row, ceil(S / 4); K, total_slabs and spp count the slots
  MnvFastDiv d_per_row, d_R;
  struct Res {
    mnv_rsrc a, b;
    const unsigned* tab;  // LDS: [total_slabs * 4][2]
  };
  static bool takes(int S) { return S >= 4 && (S % 4 == 0 || (S % 4 == 3 && S >= 7)); }
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(bottom, (unsigned)(g.N * g.C * g.HW) * 4u);
    r.b = mnv_make_rsrc(filter, (unsigned)(g.K * g.CRS) * 4u);
    r.tab = nullptr;
  }
  size_t extra_lds_bytes() const { return (size_t)total_slabs * 8 * sizeof(unsigned); }
  __device__ void block_init(Res& r, float* extra, int, int) const {
    unsigned* tab = reinterpret_cast<unsigned*>(extra);
    r.tab = tab;
    for (int i = threadIdx.x; i < total_slabs * 4; i += blockDim.x) {
      const int row = mnv_fastdiv(i, d_per_row), q = i - row * per_row;  // filter row (c, r'), group in it
      const int c = mnv_fastdiv(row, d_R), rp = row - c * g.R;
      const int first = q == per_row - 1 ? g.S - 4 : 4 * q;            // the group's first tap s'
      const unsigned pixel = (unsigned)(c * g.HW + (g.R - 1 - rp) * g.W + g.S - 4 - first) * 4u;
      tab[2 * i] = i < groups ? pixel : MNV_OOB;
      tab[2 * i + 1] = i < groups ? (unsigned)(row * g.S + first) * 4u : MNV_OOB;
    }
  }
  __device__ void a_init(const Res&, AState&, int) const {}
  __device__ void b_init(const Res&, BState&, int) const {}
  __device__ void a_load(const Res& r, const AState&, const unsigned (&off)[1], int period, int s, int kl,
                         float (&v)[4]) const {
    const unsigned t = r.tab[2 * ((period * spp + s) * 4 + (kl >> 2))];
    const unsigned one[1] = {off[0] + t};
    mnv_fetch_vec<1>(r.a, one, 0, v);
  }
  // What a row's last group has to clear is cleared on the way to LDS, and the filter's vector is reversed
  // there: made where it is loaded, every step waited for its own loads (256 images of 3 x 227 x 227 467 -> 432 us, 50 100 -> 96; the same bits).
  static constexpr bool A_STASH_FIX = true, B_STASH_FIX = true;
  __device__ bool cut(int period, int s, int kl) const {
    const int i = (period * spp + s) * 4 + (kl >> 2);
    return g.S % 4 != 0 && i - mnv_fastdiv(i, d_per_row) * per_row == per_row - 1;
  }
  __device__ void a_stash_fix(int period, int s, int kl, float (&v)[4]) const { v[3] = cut(period, s, kl) ? 0.f : v[3]; }
  __device__ void b_stash_fix(int period, int s, int kl, float (&v)[4]) const {
    const float first = v[0], second = v[1];
    v[0] = v[3]; v[1] = v[2]; v[2] = second;
    v[3] = cut(period, s, kl) ? 0.f : first;
  }
  __device__ void b_period(const BState&, unsigned (&off)[1], int n, int, int) const {
    off[0] = n < N ? (unsigned)(n * g.CRS) * 4u : MNV_OOB;
  }
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[1], int period, int s, int kl,
                         float (&v)[4]) const {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 t = *reinterpret_cast<const u2*>(__builtin_assume_aligned(r.tab + 2 * ((period * spp + s) * 4 + (kl >> 2)), 8));
    const unsigned one[1] = {(off[0] | t.y) & MNV_OOB ? MNV_OOB : off[0] + t.y};
    mnv_fetch_vec<1>(r.b, one, 0, v);
  }
};

// ------------------------------------------------------------ backward data
// FAST additionally means both strides are 1, so every (row, col) of the shifted window
// is a real output position.
template <bool FAST, bool PAD = false>
struct ConvBwdData {
  static constexpr bool A_KFAST = false, B_KFAST = true;
  static constexpr int A_NOFF = 4, B_NOFF = FAST ? 1 : 4;
  const float* __restrict__ top_diff;
  const float* __restrict__ filter;
  float* __restrict__ bottom_diff;
  ConvGeom g;
  int M, N, K, total_slabs, spp;  // N*H*W, C, Kout*R*S
  // fused epilogue (or null): the activations the bottom tensor went through a ReLU with;
  // bottom_diff = gate > 0 ? gradient : 0, the selection mnv_relu_bwd makes
  const float* __restrict__ gate;
  struct Res {
    mnv_rsrc a, b;
  };
  struct AState {
    int off[4], yx[4];  // image offset into top_diff; (y+ph-R+1, x+pw-S+1)
  };
  struct BState {};
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(top_diff, (unsigned)(g.N * g.K * g.HoWo) * 4u);
    r.b = mnv_make_rsrc(filter, (unsigned)(FAST ? N * g.RS * spp * 16 : g.K * g.CRS) * 4u);
  }
  __device__ void a_init(const Res& res, AState& st, int m) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int mm = m + q;
      int img = mnv_fastdiv(mm, g.d_HW);
      int pos = mm - img * g.HW;
      int y = mnv_fastdiv(pos, g.d_W);
      int x = pos - y * g.W;
      int ty0 = y + g.ph - g.R + 1, tx0 = x + g.pw - g.S + 1;
      st.off[q] = img * g.K * g.HoWo + (FAST ? ty0 * g.Wo + tx0 : 0);
      st.yx[q] = mm < M ? pack_yx(ty0, tx0) : pack_yx(MNV_FAR, MNV_FAR);
    }
  }
  __device__ void b_init(const Res&, BState&, int) const {}
  __device__ void a_period(const AState& st, unsigned (&off)[4], int, int kl, int period) const {
    if (FAST) {  // period = tap (r', s'), kl = output channel within the slab
      int rp = mnv_fastdiv(period, g.d_S);
      int sp = period - rp * g.S;
      int koff = kl * g.HoWo + rp * g.Wo + sp;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int i = unpack_y(st.yx[q]) + rp, j = unpack_x(st.yx[q]) + sp;
        bool ok = ((unsigned)i < (unsigned)g.Ho) & ((unsigned)j < (unsigned)g.Wo);
        off[q] = ok ? (unsigned)(st.off[q] + koff) * 4u : MNV_OOB;
      }
    } else {  // flat k = (ko, r', s')
      int k = period * 16 + kl;
      int ko = mnv_fastdiv(k, g.d_RS);
      int rs = k - ko * g.RS;
      int rp = mnv_fastdiv(rs, g.d_S);
      int sp = rs - rp * g.S;
      int koff = ko * g.HoWo;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int ty = unpack_y(st.yx[q]) + rp, tx = unpack_x(st.yx[q]) + sp;
        int tyc = ty < 0 ? 0 : ty, txc = tx < 0 ? 0 : tx;
        int i = mnv_fastdiv(tyc, g.d_sv), j = mnv_fastdiv(txc, g.d_sh);
        bool ok = (k < K) & (ty >= 0) & (tx >= 0) & (i * g.sv == ty) & (j * g.sh == tx) &
                  (i < g.Ho) & (j < g.Wo);
        off[q] = ok ? (unsigned)(st.off[q] + koff + i * g.Wo + j) * 4u : MNV_OOB;
      }
    }
  }
  __device__ void a_load(const Res& r, const AState&, const unsigned (&off)[4], int, int s, int kl,
                         float (&v)[4]) const {
    const unsigned slab = FAST ? (unsigned)s * 16u * (unsigned)g.HoWo * 4u : 0u;
    if (PAD) {
      const bool ok = s * 16 + kl < g.K;
      const unsigned in[4] = {ok ? off[0] : MNV_OOB, ok ? off[1] : MNV_OOB, ok ? off[2] : MNV_OOB, ok ? off[3] : MNV_OOB};
      mnv_fetch_vec<4>(r.a, in, slab, v);
    } else {
      mnv_fetch_vec<4>(r.a, off, slab, v);
    }
  }
  __device__ int channels() const { return g.K; }
  __device__ int channel_floats() const { return g.HoWo; }
  size_t extra_lds_bytes() const { return 0; }
  __device__ void block_init(Res&, float*, int, int) const {}
  // B[kk, c] = filter[ko, c, r', s'].  FAST reads the permuted copy [c][r's'][ko, padded to 16].
  __device__ void b_period(const BState&, unsigned (&off)[B_NOFF], int n, int kl,
                           int period) const {
    if (FAST) {
      off[0] = (n < N) ? (unsigned)((n * g.RS + period) * spp * 16 + kl) * 4u : MNV_OOB;
    } else {
      int k = period * 16 + kl;
      int ko = mnv_fastdiv(k, g.d_RS);
      int rs = k - ko * g.RS;
#pragma unroll
      for (int q = 0; q < B_NOFF; ++q) {
        bool ok = (n < N) & (k + q < K);
        off[q] = ok ? (unsigned)(ko * g.CRS + n * g.RS + rs) * 4u : MNV_OOB;
        ++rs;
        bool wrap = rs == g.RS;
        rs = wrap ? 0 : rs;
        ko += wrap ? 1 : 0;
      }
    }
  }
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[B_NOFF], int, int s,
                         int, float (&v)[4]) const {
    mnv_fetch_vec<B_NOFF>(r.b, off, FAST ? (unsigned)s * 64u : 0u, v);
  }
  __device__ void c_store(int m, int n, float x) const {
    int img = mnv_fastdiv(m, g.d_HW);
    int pos = m - img * g.HW;
    const size_t at = ((size_t)img * N + n) * g.HW + pos;
    if (gate) x = gate[at] > 0.f ? x : 0.f;
    bottom_diff[at] = x;
  }
  static constexpr bool C_STORE4 = true;
  __device__ void c_store4(int m, int n, const float (&x)[4]) const {
    int img = mnv_fastdiv(m, g.d_HW);
    int pos = m - img * g.HW;
    if (m + 3 < M && pos + 3 < g.HW) {
      const size_t at = ((size_t)img * N + n) * g.HW + pos;
      mnv_f4u v = {x[0], x[1], x[2], x[3]};
      if (gate) {
        const mnv_f4u t = *reinterpret_cast<const mnv_f4u*>(gate + at);
        v.x = t.x > 0.f ? v.x : 0.f; v.y = t.y > 0.f ? v.y : 0.f;
        v.z = t.z > 0.f ? v.z : 0.f; v.w = t.w > 0.f ? v.w : 0.f;
      }
      *reinterpret_cast<mnv_f4u*>(bottom_diff + at) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (m + q < M) c_store(m + q, n, x[q]);
    }
  }
};

// Strides above 1.  An input position is met by the filter taps of one class modulo the stride per dimension
// only, 1 / (sv sh) of them; the generic policy multiplies all, zeros but for that share.  Here the positions are
// taken class by class ("phase"): each is a product of its own, the unit-stride correlation of top_diff with
// every sv-th row and sh-th column of the filter, and all of them are one launch, those with the most taps first.
// Row class rho = 0 .. sv - 1 meets the taps r' = rho + sv t (R-1-r of the filter); its rows are y = a + sv u
// with a = (R - 1 - ph - rho) mod sv, and they meet output row u + i0 + t.  Columns likewise.  Where a stride is beyond the
// plane, only the classes with a position are taken, by a: stride 20 over 2 x 2 planes has 4 phases, not 400.  Every phase has
// `phase_rows` rows of the product, (image, u, v) and what fills up to whole tiles; rows past a phase's own read 0
// and are not stored.  `filter` is the permuted copy [c][taps, phase by phase][k, padded to 16] (PAD as above).
// What bounds it is what bounds the unit-stride gathers (a trip to memory per slab on the small tiles), and the stores,
// which leave every sh-th float of a row.
template <bool PAD>
struct ConvBwdDataPhases {
  static constexpr bool A_KFAST = false, B_KFAST = true, PHASED = true, PADDED = PAD;
  static constexpr int A_NOFF = 4, B_NOFF = 1;
  const float* __restrict__ top_diff;
  const float* __restrict__ filter;
  float* __restrict__ bottom_diff;
  ConvGeom g;
  int M, N, total_slabs, spp;      // phases * phase_rows, C, most taps of a phase * spp
  const float* __restrict__ gate;  // as in ConvBwdData
  int phase_rows;
  // of class 0: its first row / column, and the output row / column that this one meets with its first tap
  int a0, b0, i00, j00;
  // H, W, R, S = stride * quotient + rest: the first `rest` classes have one row, column, tap more
  int hq, hr, wq, wr, rq, rr, sq, sr;
  int col_classes;  // phases = row classes * col_classes
  MnvFastDiv d_cols, d_rows, d_plane[4], d_width[2], d_taps[2];  // by [rows more * 2 + columns more], [columns more], [taps more]
  struct Phase {
    int a, b, i0, j0, rows_more, cols_more, taps, taps_per_row, tap0;
    MnvFastDiv d_taps_per_row;
  };
  struct Res {
    mnv_rsrc a, b;
    Phase ph;
    int row0, end;  // the phase's own rows of the product
  };
  struct AState {
    int off[4], yx[4], taps_per_row;
    MnvFastDiv d_taps_per_row;
  };
  struct BState {
    unsigned off;
  };
  __device__ Phase phase(int q) const {
    int rho = mnv_fastdiv(q, d_cols), sigma = q - rho * col_classes;
    if (g.sv > g.H) rho = rho <= a0 ? a0 - rho : a0 - rho + g.sv;
    if (g.sh > g.W) sigma = sigma <= b0 ? b0 - sigma : b0 - sigma + g.sh;
    Phase p;
    p.a = a0 - rho;
    p.i0 = i00;
    if (p.a < 0) p.a += g.sv, ++p.i0;
    p.b = b0 - sigma;
    p.j0 = j00;
    if (p.b < 0) p.b += g.sh, ++p.j0;
    p.rows_more = p.a < hr;
    p.cols_more = p.b < wr;
    const int taps_per_column = rq + (rho < rr);
    p.taps_per_row = sq + (sigma < sr);
    p.taps = taps_per_column * p.taps_per_row;
    p.tap0 = (rho * rq + (rho < rr ? rho : rr)) * g.S + taps_per_column * (sigma * sq + (sigma < sr ? sigma : sr));
    p.d_taps_per_row = sigma < sr ? d_taps[1] : d_taps[0];
    return p;
  }
  __device__ int rows(const Phase& p) const { return g.N * (hq + p.rows_more) * (wq + p.cols_more); }
  __device__ int phase_slabs(int m0) const {
    const int q = mnv_fastdiv(m0, d_rows);
    const Phase p = phase(q);
    return m0 - q * phase_rows < rows(p) ? p.taps * spp : 0;
  }
  // (image, u, v) of a row of the phase
  __device__ void place(const Phase& p, int row, int& img, int& u, int& v) const {
    const int w = wq + p.cols_more;
    img = mnv_fastdiv(row, p.rows_more ? (p.cols_more ? d_plane[3] : d_plane[2]) : p.cols_more ? d_plane[1] : d_plane[0]);
    const int pos = row - img * (hq + p.rows_more) * w;
    u = mnv_fastdiv(pos, p.cols_more ? d_width[1] : d_width[0]);
    v = pos - u * w;
  }
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(top_diff, (unsigned)(g.N * g.K * g.HoWo) * 4u);
    r.b = mnv_make_rsrc(filter, (unsigned)(N * g.RS * spp * 16) * 4u);
  }
  __device__ int channels() const { return g.K; }
  __device__ int channel_floats() const { return g.HoWo; }
  size_t extra_lds_bytes() const { return 0; }
  __device__ void block_init(Res& r, float*, int m0, int) const {
    const int q = mnv_fastdiv(m0, d_rows);
    r.ph = phase(q);
    r.row0 = q * phase_rows;
    r.end = r.row0 + rows(r.ph);
  }
  __device__ void a_init(const Res& r, AState& st, int m) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int img, u, v;
      place(r.ph, m + q - r.row0, img, u, v);
      const int i = u + r.ph.i0, j = v + r.ph.j0;
      st.off[q] = img * g.K * g.HoWo + i * g.Wo + j;
      st.yx[q] = m + q < r.end ? pack_yx(i, j) : pack_yx(MNV_FAR, MNV_FAR);
    }
    st.taps_per_row = r.ph.taps_per_row;
    st.d_taps_per_row = r.ph.d_taps_per_row;
  }
  __device__ void b_init(const Res& r, BState& st, int n) const {
    st.off = n < N ? (unsigned)((n * g.RS + r.ph.tap0) * spp * 16) * 4u : MNV_OOB;
  }
  // period = tap of the phase, kl = output channel within the slab
  __device__ void a_period(const AState& st, unsigned (&off)[4], int, int kl, int period) const {
    const int rp = mnv_fastdiv(period, st.d_taps_per_row), sp = period - rp * st.taps_per_row;
    const int koff = kl * g.HoWo + rp * g.Wo + sp;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = unpack_y(st.yx[q]) + rp, j = unpack_x(st.yx[q]) + sp;
      const bool ok = ((unsigned)i < (unsigned)g.Ho) & ((unsigned)j < (unsigned)g.Wo);
      off[q] = ok ? (unsigned)(st.off[q] + koff) * 4u : MNV_OOB;
    }
  }
  __device__ void a_load(const Res& r, const AState&, const unsigned (&off)[4], int, int s, int kl, float (&v)[4]) const {
    const unsigned slab = (unsigned)s * 16u * (unsigned)g.HoWo * 4u;
    if (PAD) {
      const bool ok = s * 16 + kl < g.K;
      const unsigned in[4] = {ok ? off[0] : MNV_OOB, ok ? off[1] : MNV_OOB, ok ? off[2] : MNV_OOB, ok ? off[3] : MNV_OOB};
      mnv_fetch_vec<4>(r.a, in, slab, v);
    } else {
      mnv_fetch_vec<4>(r.a, off, slab, v);
    }
  }
  __device__ void b_period(const BState& st, unsigned (&off)[1], int, int kl, int period) const {
    off[0] = st.off + (unsigned)(period * spp * 16 + kl) * 4u;  // past the filter for MNV_OOB
  }
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[1], int, int s, int, float (&v)[4]) const {
    mnv_fetch_vec<1>(r.b, off, (unsigned)s * 64u, v);
  }
  __device__ void c_store(int m, int n, float x) const {
    const int q = mnv_fastdiv(m, d_rows), row = m - q * phase_rows;
    const Phase p = phase(q);
    if (row >= rows(p)) return;
    int img, u, v;
    place(p, row, img, u, v);
    const size_t at = ((size_t)img * N + n) * g.HW + (p.a + g.sv * u) * g.W + p.b + g.sh * v;
    if (gate) x = gate[at] > 0.f ? x : 0.f;
    bottom_diff[at] = x;
  }
};

// The fast gathers of B, four channels of one position to a vector: for mnv_gemm_small_kernel.
template <class B, bool PAD>
struct ConvOneRow : B {
  typedef B StoredBy;
  static constexpr bool A_KFAST = true;
  static constexpr int A_NOFF = 1;
  __device__ void a_period(const typename B::AState& st, unsigned (&off)[1], int m, int kl, int period) const {
    unsigned rows[4];  // of m and the three rows after it, which are not used
    B::a_period(st, rows, m, kl, period);
    off[0] = rows[0];
  }
  __device__ void a_load(const typename B::Res& r, const typename B::AState&, const unsigned (&off)[1], int, int s, int kl,
                         float (&v)[4]) const {
    const unsigned plane = (unsigned)this->channel_floats() * 4u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned at = !PAD || s * 16 + kl + q < this->channels() ? off[0] : MNV_OOB;
      v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r.a, (int)at, (int)((unsigned)(s * 16 + q) * plane), 0));
    }
  }
};

// ---------------------------------------------------------- backward filter
struct ConvBwdFilter {
  static constexpr bool A_KFAST = true, B_KFAST = true;
  static constexpr int A_NOFF = 4, B_NOFF = 4;
  const float* __restrict__ bottom;
  const float* __restrict__ top_diff;
  float* __restrict__ filter_diff;
  ConvGeom g;
  int M, N, K, total_slabs, spp;  // C*R*S, Kout, N*Ho*Wo
  int accumulate;                 // filter_diff += (a later chunk of images)
  // Parameter update in the store: filter_diff receives sgd_w - sgd_scale * gradient
  // (sgd_w may be filter_diff itself)
  const float* sgd_w;
  float sgd_scale;
  struct Res {
    mnv_rsrc a, b;
  };
  struct AState {
    int off, dyx;  // c*H*W + dy*W + dx ; (dy, dx) = (R-1-r'-ph, S-1-s'-pw)
  };
  struct BState {};
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(bottom, (unsigned)(g.N * g.C * g.HW) * 4u);
    r.b = mnv_make_rsrc(top_diff, (unsigned)(g.N * g.K * g.HoWo) * 4u);
  }
  __device__ void a_init(const Res& res, AState& st, int m) const {
    int c = mnv_fastdiv(m, g.d_RS);
    int rs = m - c * g.RS;
    int rp = mnv_fastdiv(rs, g.d_S);
    int sp = rs - rp * g.S;
    int dy = g.R - 1 - rp - g.ph, dx = g.S - 1 - sp - g.pw;
    st.off = c * g.HW + dy * g.W + dx;
    st.dyx = m < M ? pack_yx(dy, dx) : pack_yx(MNV_FAR, MNV_FAR);
  }
  __device__ void b_init(const Res&, BState&, int) const {}
  // A[m, kk..kk+3] = bottom[img, c, i*sv + dy, j*sh + dx] for kk = (img, i, j)
  __device__ void a_period(const AState& st, unsigned (&off)[4], int, int kl, int period) const {
    int k = period * 16 + kl;
    int img = mnv_fastdiv(k, g.d_HoWo);
    int pos = k - img * g.HoWo;
    int i = mnv_fastdiv(pos, g.d_Wo);
    int j = pos - i * g.Wo;
    const int dy = unpack_y(st.dyx), dx = unpack_x(st.dyx);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int y = i * g.sv + dy, x = j * g.sh + dx;
      bool ok = (k + q < K) & ((unsigned)y < (unsigned)g.H) & ((unsigned)x < (unsigned)g.W);
      unsigned o = (unsigned)(img * g.C * g.HW + st.off + i * g.sv * g.W + j * g.sh) * 4u;
      off[q] = ok ? o : MNV_OOB;
      ++j;
      bool wj = j == g.Wo;
      j = wj ? 0 : j;
      i += wj ? 1 : 0;
      bool wi = i == g.Ho;
      i = wi ? 0 : i;
      img += wi ? 1 : 0;
    }
  }
  __device__ void a_load(const Res& r, const AState&, const unsigned (&off)[4], int, int, int,
                         float (&v)[4]) const {
    mnv_fetch_vec<4>(r.a, off, 0u, v);
  }
  size_t extra_lds_bytes() const { return 0; }
  __device__ void block_init(Res&, float*, int, int) const {}
  // B[kk..kk+3, ko] = top_diff[img, ko, i, j]
  __device__ void b_period(const BState&, unsigned (&off)[4], int n, int kl, int period) const {
    int k = period * 16 + kl;
    int img = mnv_fastdiv(k, g.d_HoWo);
    int pos = k - img * g.HoWo;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bool ok = (n < N) & (k + q < K);
      off[q] = ok ? (unsigned)((img * N + n) * g.HoWo + pos) * 4u : MNV_OOB;
      ++pos;
      bool wrap = pos == g.HoWo;
      pos = wrap ? 0 : pos;
      img += wrap ? 1 : 0;
    }
  }
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[4], int, int, int,
                         float (&v)[4]) const {
    mnv_fetch_vec<4>(r.b, off, 0u, v);
  }
  __device__ void c_store(int m, int n, float x) const {
    const size_t at = (size_t)n * M + m;
    if (sgd_w) x = sgd_w[at] - sgd_scale * x;
    else if (accumulate) x = filter_diff[at] + x;
    filter_diff[at] = x;
  }
};

// Filter gradient, fast addressing.  The GEMM rows are ordered (tap, channel) instead of
// (channel, tap), so a thread's tap is fixed and the only thing that changes from slab to
// slab is which 16 output positions are reduced.  The reduction runs image by image
// (one period per image, positions padded to a multiple of 16).  A workgroup first writes,
// for every tap its rows touch, a table pos -> byte offset of the input pixel that the tap
// pairs with output position pos (or MNV_OOB when that pixel is padding or pos is past the
// image); a slab's im2col offsets are then one 16-byte LDS read and four adds per vector.
// top_diff is read with 16-byte loads of 4 consecutive positions; only the last, partial
// slab of an image needs per-element masking.
//
// NP ("no padding", any channel count): with ph == pw == 0 every tap of every output
// position is a real pixel, so the pixel offset splits into a row part (channel, tap) and a
// position part: one position table serves all rows, which stay in (channel, tap) order.
//
// LK (padded convolutions whose channel count is a multiple of 16, so that every 16 rows of
// a tile are 16 consecutive channels of one tap): the gathered operand is fetched with the
// slab's 16 positions on 16 consecutive lanes.  A load instruction then reads 64 contiguous
// bytes of each of four channel planes instead of 16 bytes of each of sixteen; a thread's
// eight rows are 16 rows apart, so what distinguishes them (tap, first channel) is uniform
// and lives in the workgroup's Res; and nothing else changes: same tile in LDS, same
// products, same order.  LK = 1: all rows of a tile share one tap (channel counts that are
// multiples of 128: one table entry and one add per thread and slab); LK = 2: a table entry
// per row group; LK = 3: the rows of a tile lie in at most two taps (96 channels: conv2 of the
// AlexNet shape), so a thread reads two table entries per slab and every row group picks one
// of the two by a uniform flag.  Row groups past M fetch whatever their offsets point at: their
// accumulators are never stored.
template <bool NP, int LK = 0>
struct ConvBwdFilterFast {
  static constexpr bool A_KFAST = true, B_KFAST = true;
  static constexpr bool A_LANE_K = LK != 0;
  static constexpr int A_NOFF = 1, B_NOFF = 1;
  const float* __restrict__ bottom;
  const float* __restrict__ top_diff;
  float* __restrict__ filter_diff;
  ConvGeom g;
  int M, N, K, total_slabs, spp;  // C*R*S rows in (tap, c) order, Kout, N*Ho*Wo
  int PP, taps_per_block;         // padded positions per image, table rows per workgroup
  MnvFastDiv d_C;
  int accumulate;                 // filter_diff += (a later chunk of images)
  const float* sgd_w;             // update in the store, as in ConvBwdFilter
  float sgd_scale;
  struct Res {
    mnv_rsrc a, b;
    const unsigned* tab;  // LDS: [taps_per_block][PP]
    int tap0;             // first tap of the workgroup's rows
    // LK: row group j (rows m0 + 16 j ...) starts at channel c0: c0 * H * W * 4, its table
    // row (tap - tap0) * PP, and whether it lies inside M
    unsigned group_off[LK ? 8 : 1];
    int group_trow[LK ? 8 : 1];
    bool group_ok[LK ? 8 : 1];
    bool group_second[LK ? 8 : 1];  // LK = 3: the group's rows lie in the tile's second tap
  };
  struct AState {
    unsigned cbase;  // c*H*W*4, or MNV_OOB for rows past M
    int trow;        // (tap - first tap of the workgroup) * PP
  };
  struct BState {};
  __device__ void make_res(Res& r) const {
    r.a = mnv_make_rsrc(bottom, (unsigned)(g.N * g.C * g.HW) * 4u);
    r.b = mnv_make_rsrc(top_diff, (unsigned)(g.N * g.K * g.HoWo) * 4u);
    r.tab = nullptr;
    r.tap0 = 0;
  }
  size_t extra_lds_bytes() const { return (size_t)taps_per_block * PP * sizeof(unsigned); }
  __device__ void block_init(Res& r, float* extra, int m0, int) const {
    unsigned* tab = reinterpret_cast<unsigned*>(extra);
    r.tab = tab;
    const int tap0 = mnv_fastdiv(m0, d_C);
    r.tap0 = tap0;
    if (LK) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int row = m0 + 16 * j, tap = mnv_fastdiv(row, d_C);
        r.group_off[j] = (unsigned)((row - tap * g.C) * g.HW) * 4u;
        r.group_trow[j] = (tap - tap0 < taps_per_block ? tap - tap0 : 0) * PP;
        r.group_ok[j] = row < M;
        r.group_second[j] = tap - tap0 == 1;
      }
    }
    for (int e = threadIdx.x; e < taps_per_block * PP; e += blockDim.x) {
      int t = e / PP, pos = e - t * PP;
      int tap = tap0 + t;
      int rp = mnv_fastdiv(tap, g.d_S), sp = tap - rp * g.S;
      int dy = NP ? 0 : g.R - 1 - rp - g.ph, dx = NP ? 0 : g.S - 1 - sp - g.pw;
      int i = mnv_fastdiv(pos, g.d_Wo), j = pos - i * g.Wo;
      int y = i * g.sv + dy, x = j * g.sh + dx;
      bool ok = (pos < g.HoWo) & (NP | (tap < g.RS)) & ((unsigned)y < (unsigned)g.H) &
                ((unsigned)x < (unsigned)g.W);
      tab[e] = ok ? (unsigned)(y * g.W + x) * 4u : MNV_OOB;
    }
  }
  __device__ void a_init(const Res& res, AState& st, int m) const {
    if (NP) {  // m = (c, r', s'); the tap's shift is part of the row offset
      int c = mnv_fastdiv(m, g.d_RS);
      int rs = m - c * g.RS;
      int rp = mnv_fastdiv(rs, g.d_S), sp = rs - rp * g.S;
      st.cbase = m < M ? (unsigned)(c * g.HW + (g.R - 1 - rp) * g.W + (g.S - 1 - sp)) * 4u : MNV_OOB;
      st.trow = 0;
      return;
    }
    if (LK) {  // the thread's row inside its groups of 16: a channel offset
      st.cbase = (unsigned)((m & 15) * g.HW) * 4u;
      st.trow = 0;
      return;
    }
    int tap = mnv_fastdiv(m, d_C);
    int c = m - tap * g.C;
    st.cbase = m < M ? (unsigned)(c * g.HW) * 4u : MNV_OOB;
    int t = tap - res.tap0;
    st.trow = (t < taps_per_block ? t : 0) * PP;  // rows past M read a valid table row; cbase masks them
  }
  __device__ void b_init(const Res&, BState&, int) const {}
  // off[0]: byte offset of the vector's entries of slab 0 in the table (the pixel offsets
  // come from the table every slab); a slab then adds s * 64 to it, one instruction
  __device__ void a_period(const AState& st, unsigned (&off)[1], int, int kl, int) const {
    off[0] = (unsigned)(st.trow + kl) * 4u;
  }
  template <int AV>
  __device__ void a_load_lanek(const Res& r, const AState& st, int period, int s, int kl,
                               float (&v)[AV][4]) const {
    static_assert(AV * 4 <= 8, "row groups of a tile");
    const unsigned img = (unsigned)period * (unsigned)(g.C * g.HW) * 4u;
    const int pos = s * 16 + kl;
    const unsigned one = st.cbase + r.tab[pos];
    const unsigned two = LK == 3 ? st.cbase + r.tab[PP + pos] : 0u;
#pragma unroll
    for (int j = 0; j < AV * 4; ++j) {
      unsigned voff = one;
      if (LK == 3) voff = r.group_second[j] ? two : one;
      if (LK == 2) {
        voff = st.cbase + r.tab[r.group_trow[j] + pos];
        voff = r.group_ok[j] ? voff : MNV_OOB;
      }
      v[j / 4][j % 4] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(r.a, (int)voff, (int)(img + r.group_off[j]), 0));
    }
  }
  __device__ void a_load(const Res& r, const AState& st, const unsigned (&off)[1], int period, int s,
                         int, float (&v)[4]) const {
    // the four entries are one aligned 16-byte LDS read: rows are PP (a multiple of 16)
    // entries long and kl is a multiple of 4
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const u4 t = *reinterpret_cast<const u4*>(__builtin_assume_aligned(
        reinterpret_cast<const char*>(r.tab) + (off[0] + (unsigned)s * 64u), 16));
    const unsigned soff = (unsigned)period * (unsigned)(g.C * g.HW) * 4u;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                           r.a, (int)(st.cbase + t[q]), (int)soff, 0));
  }
  __device__ void b_period(const BState&, unsigned (&off)[1], int n, int kl, int) const {
    off[0] = n < N ? (unsigned)(n * g.HoWo + kl) * 4u : MNV_OOB;
  }
  // Every slab is one 16-byte load per vector.  In the last slab of an image the positions
  // past the image read whatever follows in memory (the next plane, or 0 past the tensor);
  // b_stash_fix zeroes them on their way to LDS, when the values have arrived anyway.  (A
  // branch to per-element loads at this point made the wavefront wait for every load in
  // flight, the gathered operand's just-issued ones included, once per image.)
  static constexpr bool B_STASH_FIX = true;
  __device__ void b_load(const Res& r, const BState&, const unsigned (&off)[1], int period, int s,
                         int, float (&v)[4]) const {
    const unsigned soff = ((unsigned)period * (unsigned)(g.K * g.HoWo) + (unsigned)s * 16u) * 4u;
    mnv_fetch_vec<1>(r.b, off, soff, v);
  }
  __device__ void b_stash_fix(int, int s, int kl, float (&v)[4]) const {
    if (s * 16 + 16 > g.HoWo) {  // uniform
      const int first = s * 16 + kl;
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = first + q < g.HoWo ? v[q] : 0.f;
    }
  }
  __device__ void c_store(int m, int n, float x) const {
    int row = m;
    if (!NP) {
      int tap = mnv_fastdiv(m, d_C);
      row = (m - tap * g.C) * g.RS + tap;
    }
    const size_t at = (size_t)n * M + row;
    if (sgd_w) x = sgd_w[at] - sgd_scale * x;
    else if (accumulate) x = filter_diff[at] + x;
    filter_diff[at] = x;
  }
};

// Filter permutations for the FAST policies (a few MB at most, one pass); the last dimension is
// padded with zeros to `width`:
//   to_rsc: out[k][r's'][c] = in[k][c][r's']      (forward)
//   to_crk: out[c][r's'][k] = in[k][c][r's']      (data gradient; with strides above 1 the taps class by
//           class of (r' mod sv, s' mod sh), see ConvBwdDataPhases)
__global__ __launch_bounds__(256) void mnv_filter_permute_kernel(const float* __restrict__ in,
                                                                 float* __restrict__ out, int K,
                                                                 int C, int R, int S, int width, bool to_crk, int sv, int sh) {
  const int RS = R * S, total = (to_crk ? C : K) * RS * width;
  for (int o = blockIdx.x * 256 + threadIdx.x; o < total; o += gridDim.x * 256) {
    const int last = o % width, first = o / (width * RS);
    int rs = (o / width) % RS;
    if (sv > 1 || sh > 1) {
      int rho = 0, sigma = 0, rows = (R - 1) / sv + 1, cols = (S - 1) / sh + 1;
      while (rs >= rows * S) rs -= rows * S, ++rho, rows = (R - rho - 1) / sv + 1;
      while (rs >= rows * cols) rs -= rows * cols, ++sigma, cols = (S - sigma - 1) / sh + 1;
      rs = (rho + sv * (rs / cols)) * S + sigma + sh * (rs % cols);
    }
    const int k = to_crk ? last : first, c = to_crk ? first : last;
    out[o] = last < (to_crk ? K : C) ? in[(k * C + c) * RS + rs] : 0.f;
  }
}

int permute_filter(const float* in, float* out, int K, int C, int R, int S, int width, bool to_crk, hipStream_t s,
                   int sv = 1, int sh = 1) {
  int total = (to_crk ? C : K) * R * S * width;
  int blocks = (total + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(mnv_filter_permute_kernel, dim3(blocks), dim3(256), 0, s, in, out, K, C, R, S, width, to_crk, sv, sh);
  return MNV_LAUNCH_STATUS();
}

typedef MnvGemmTile<128, 128, 16, 2, 2> TileBig;
typedef MnvGemmTile<64, 64, 16, 2, 2> TileSmall;
typedef MnvGemmTile<128, 128, 16, 4, 1, 0, 96> Tile96;  // four wavefronts of 32 x 96
// Four wavefronts of 32 x 32 for outputs of at most 32 columns (a convolution with few
// output channels): a 64-column tile would spend half or more of its multiplies on padding.
// 64 columns are staged because a slab of 32 would not give every thread a vector to fetch.
typedef MnvGemmTile<128, 64, 16, 4, 1, 0, 32> TileThin;

// tile 0: 64x64 output tiles, tile 1: 128x128, tile 2: 128x96, tile 3: 128x32
const int kTileM[4] = {64, 128, 128, 128}, kTileN[4] = {64, 128, 96, 32};
// Eight wavefronts of 64 x 64 (512 threads, two workgroups per CU): a quarter fewer bytes
// fetched and staged per multiply than TileBig, and every element summed in the same order.
// For the (tap, channel) forward and data-gradient policies, when the 256 x 128 tiles fill
// the chip's two-per-CU slots in whole rounds to 97% (conv3 / conv4 forward and conv4 / conv5
// data gradient of the AlexNet shape at batch 256: 507 tiles on 512 slots, 2-3% faster; conv2
// forward, 1458 tiles in three rounds of 512 at 95%, is 3% SLOWER than on 128 x 128 tiles with
// their cut tail).
typedef MnvGemmTile<256, 128, 16, 4, 2> TileTall;
// What the plan queries of the forward pass and the data gradient report; a launch that is given one launches nothing.
struct DirectPlan {
  int rows, ranges, parts, classes = 1;  // rows of the tile (0: minimal filtering), k ranges, in bf16 parts, products of one launch
};
int report(DirectPlan* plan, int rows, int ranges, int parts) {
  plan->rows = rows;
  plan->ranges = ranges;
  plan->parts = parts;
  return MNV_OK;
}
template <class P>
int launch_tile(int tile, const P& p, int splits, void* ws, hipStream_t s, size_t tail_bytes = 0, DirectPlan* plan = nullptr) {
  if constexpr (P::A_KFAST == false && P::B_NOFF == 1 && !MnvPhased<P>::value) {
    if (tile == 1 && splits == 1) {
      const long long tiles = (long long)((p.M + 255) / 256) * ((p.N + 127) / 128);
      const long long slots = 2LL * mnv_cu_count(), rounds = (tiles + slots - 1) / slots;
      if ((double)p.M * p.N >= 0.97 * (double)(rounds * slots) * 256.0 * 128.0)
        return plan ? report(plan, 256, 1, 0) : mnv_gemm_launch<TileTall>(p, 1, ws, s);
    }
  }
  if (plan) return report(plan, kTileM[tile], splits, 0);
  switch (tile) {
    case 0: return mnv_gemm_launch<TileSmall>(p, splits, ws, s);
    case 2: return mnv_gemm_launch<Tile96>(p, splits, ws, s, tail_bytes);
    case 3: return mnv_gemm_launch<TileThin>(p, splits, ws, s);
    default: return mnv_gemm_launch<TileBig>(p, splits, ws, s, tail_bytes);
  }
}
// In bf16 parts.  128 x 128 tiles with a CU to themselves: the gathers' offsets need the registers
// (four 4-byte loads per vector; on the tile with two workgroups per CU they spill, 490 against
// 415 us for 96 -> 256 channels under 5 x 5 filters on 64 x 27 x 27).  96-column tiles: two
// workgroups of four wavefronts per CU.
typedef MnvSplitTile<128, 128, 2, 4, 2> SplitOne;
typedef MnvSplitTile<128, 128, 2, 4, 1> SplitPair;
typedef MnvSplitTile<128, 96, 2, 2, 1> Split96;

// The filter gradient: few output tiles and a very long k.  On the large tiles it runs as
// one launch of as many workgroups as the chip holds, every one with the same number of
// k-slabs (stream-k: aligned k ranges of every tile, the rest in shares; see mnv_gemm_kernel),
// when the workspace holds the partial tiles; otherwise, and on the small tiles, in `splits`
// whole k ranges.
// Slabs the filter gradient's loads run ahead (see mnv_gemm_kernel): two, which costs a
// fourth workgroup per CU.  Measured on the four padded convolutions of the AlexNet shape
// with the aligned plan: one slab ahead and four workgroups per CU 3.88 ms over the four
// launches, two ahead and three per CU 3.84 ms.
#ifndef MNV_SK_PF
#define MNV_SK_PF 2
#endif
// `plan` (optional): nothing is launched; plan[0] = rows of the tile, plan[1] = k ranges,
// plan[2] = workgroups of the stream-k launch (0: k ranges).
// `parts`: in bf16 parts where the workspace holds the partial tiles (unpadded layers, whose
// gathered operand comes four k at a time; of the padded ones, one k per lane, the fetch by fours and the cut
// together take what the faster instruction gains: 53 -> 46 us for 256 -> 384 under 3 x 3 on
// 10 x 13 x 13, 60 -> 59 for 384 -> 384, 129 -> 143 for 128 -> 256 on 32 x 56 x 56 at stride 2).  3 -> 96
// under 11 x 11, stride 4, 256 / 50 / 10 images of 227 x 227: 537 -> 386, 101 -> 89, 38 -> 34 us; 256 ->
// 256 under 1 x 1 on 16 x 28 x 28 40 -> 30.
// `small(&done)`: the launch on the small tiles, for what does not run in equal shares.
template <bool PARTS = false, class P, class Small>
int launch_filter_gradient(int tile, const P& p, int splits, void* ws, size_t ws_bytes, hipStream_t s,
                           int* plan, const Small& small) {
  if (plan) {
    plan[0] = kTileM[tile];
    plan[1] = splits;
    plan[2] = 0;
  }
  if (tile == 1 || tile == 2) {
    bool done = false;
    int* wgs = plan ? plan + 2 : nullptr;
    int rc = MNV_OK;
    if constexpr (PARTS) {
      // Few tiles have long ranges, which the pair works off faster (96 -> 256 under 3 x 3 on 64 x 28 x
      // 28, 14 tiles: 146 us, 152 with one workgroup per CU); many need twice the partial tiles for it
      // (22 -> 1408 under 5 x 5 on 17 x 17 x 17, 55 tiles: 54 and 53), and short ranges do not
      // repay twice the workgroups at all.
      const bool pair = (long long)((p.M + 127) / 128) * ((p.N + 127) / 128) < 32;
      if (tile == 2) rc = mnv_gemm_streamk_launch<Split96>(p, ws, ws_bytes, s, &done, wgs);
      else if (pair) rc = mnv_gemm_streamk_launch<SplitPair>(p, ws, ws_bytes, s, &done, wgs);
      if (!rc && !done && tile == 1) rc = mnv_gemm_streamk_launch<SplitOne>(p, ws, ws_bytes, s, &done, wgs);
    }
    if (!rc && !done) rc = tile == 1 ? mnv_gemm_streamk_launch<TileBig, MNV_SK_PF>(p, ws, ws_bytes, s, &done, wgs)
                                   : mnv_gemm_streamk_launch<Tile96, MNV_SK_PF>(p, ws, ws_bytes, s, &done, wgs);
    if (rc || done) {
      if (plan && done) plan[1] = 1;
      return rc;
    }
  }
  bool done = false;
  const int rc = small(&done);
  if (rc || done || plan) return rc;
  return launch_tile(tile, p, splits, ws, s);
}

// 128-row tiles: 96 columns wide when that leaves clearly fewer idle columns than 128
// (an output 96 or 192 wide), since the narrower tile does a little less work per byte
// staged.
int wide_tile(int n) {
  int pad128 = (n + 127) / 128 * 128, pad96 = (n + 95) / 96 * 96;
  return pad96 * 10 < pad128 * 9 ? 2 : 1;
}

// Which forward and data-gradient products run in bf16 parts, and in how many k ranges (0: not).
// From 0.7 GFLOP on where the estimate is below that of the fp32 tiles: a step of 32 k takes 1.6 us
// on SplitOne, 1.7 on Split96 alone on its CU and 1.26 of the CU's time beside another; about 3 for
// a workgroup's first loads and last stores, 4 for the reduction of the k ranges beside its bytes; the
// fp32 instruction 115 TFLOP/s on the large tiles where a CU has four of them or more (fewer as
// in mnv_pick_splits), 80 and 11 us on 64 x 64.
// us with the filter's permutation, fp32 instruction -> bf16 parts, forward: 96 -> 256 under 5 x 5 on 27 x 27,
// 1 / 2 / 10 / 64 images 27 -> 25 / 41 -> 32 / 123 -> 77 / 523 -> 415; 384 -> 384 under 3 x 3 on
// 13 x 13, 2 / 10 images 31 -> 28 / 70 -> 48; 128 -> 256 on 32 x 56 x 56 547 -> 430, stride 2 188 -> 164;
// 256 -> 256 under 1 x 1 on 16 x 28 x 28 33 -> 24; 3 -> 96 under 11 x 11, stride 4, 227 x 227, 10 / 256
// images 39 -> 35 / 555 -> 498; 64 -> 128 under 3 x 3, no padding, on 32 x 28 x 28 57 -> 35; data gradients: 96 <- 256 of 10 images 131 -> 84, 256 <- 384 54 -> 40.
// Left: 256 -> 384 of one image (0.3 GFLOP) 19 -> 21, 64 -> 128 under 1 x 1, stride 2 (0.2) 9.5 -> 10.3.
int split_ranges(int m, int n, int slabs, int tile, size_t ws_floats) {
  const double flop = 2.0 * m * n * slabs * 16.0;
  if (n <= 64 || m < 128 || flop < 7e8) return 0;
  const bool narrow = wide_tile(n) == 2;
  const long long tiles = (long long)((m + 127) / 128) * (narrow ? (n + 95) / 96 : (n + 127) / 128);
  const long long cus = mnv_cu_count();
  const size_t fit = ws_floats / ((size_t)m * n);
  static const double rate[5] = {1.0, 0.45, 0.75, 0.92, 1.0};
  const long long resident = (tiles + cus - 1) / cus;
  double best = tile == 0 ? flop / 80e6 + 11.0 : flop / 115e6 / rate[resident < 4 ? resident : 4];
  best *= 0.95;
  int z_best = 0;
  for (int z = 1; z <= 32; ++z) {
    if (z > 1 && ((size_t)z > fit || slabs / z < 4 || tiles * z > 4 * cus)) break;
    const long long per_cu = (tiles * z + cus - 1) / cus;
    const int steps = ((slabs + z - 1) / z + 1) / 2;
    double cost = narrow ? (per_cu == 1 ? 1.7 : 1.26 * per_cu) * steps + 3.0 * (double)((per_cu + 1) / 2)
                         : per_cu * (1.6 * steps + 3.0);
    if (z > 1) cost += 4.0 + 8.0 * (double)m * n * z / 6e6;
    if (cost < best * (z_best ? 0.97 : 1.0)) {
      best = cost;
      z_best = z;
    }
  }
  return z_best;
}

template <class P>
int launch_parts(const P& p, int z, void* ws, hipStream_t s, size_t ws_bytes, DirectPlan* plan = nullptr) {
  if (plan) return report(plan, 128, z, 1);
  return wide_tile(p.N) == 2 ? mnv_gemm_launch<Split96>(p, z, ws, s, ws_bytes)
                             : mnv_gemm_launch<SplitOne>(p, z, ws, s, ws_bytes);
}
// Forward and data gradient: in bf16 parts or, with `splits` k ranges, on the fp32 tile.
template <class P>
int launch_direct(int tile, const P& p, int splits, void* ws, hipStream_t s, size_t ws_bytes, DirectPlan* plan) {
  if (const int z = split_ranges(p.M, p.N, p.total_slabs, tile, ws_bytes / sizeof(float)))
    return launch_parts(p, z, ws, s, ws_bytes, plan);
  return launch_tile(tile, p, splits, ws, s, ws_bytes, plan);
}

// Bytes the large tiles' launches want for the partial tiles of a cut tail (0: no tail); `parts`: the
// policy is one that launch_direct takes.
size_t tail_workspace_bytes(int tile, int m, int n, int slabs, bool parts) {
  if (tile != 1 && tile != 2) return 0;
  const int z = parts ? split_ranges(m, n, slabs, tile, (size_t)-1) : 0;
  if (z > 1) return 0;
  const long long tiles = (long long)((m + kTileM[tile] - 1) / kTileM[tile]) * ((n + kTileN[tile] - 1) / kTileN[tile]);
  const size_t tile_floats = (size_t)kTileM[tile] * kTileN[tile];
  const MnvTailPlan t = mnv_tail_plan(tiles, slabs, tile_floats, (size_t)-1 / sizeof(float),
                                      !z ? MnvTailCost{} : tile == 2 ? Split96::TAIL : SplitOne::TAIL);
  return t.z > 1 ? (size_t)(tiles - t.begin) * t.z * tile_floats * sizeof(float) : 0;
}

// Bytes of the k ranges' partial results in bf16 parts.
size_t split_bytes(int tile, int m, int n, int slabs) {
  const int z = split_ranges(m, n, slabs, tile, (size_t)-1);
  return z > 1 ? (size_t)z * m * n * sizeof(float) : 0;
}

// Forward and data gradient on the small tiles (mnv_gemm_small_kernel) instead of `tile` with as many k ranges as it takes: the
// number of their own, 0: not.  `slabs`: of the small tiles and of the others.  A slab of a 64 x 64 or
// 128 x 32 tile takes 0.28 or 0.46 us of a CU, and 0.3 at least.  Products in bf16 parts, the more exact ones, stay.
// us: 24 -> 32 channels under 3 x 3 on 19 x 44 x 12 12.3 -> 5.8, 80 -> 32 under 5 x 5, stride 2, on 59 x 48 x 20 82 -> 36,
// data gradient 32 <- 160 under 3 x 3 on 4 x 53 x 52 34 -> 21, 40 <- 48 on 7 x 14 x 41 13.8 -> 7.7.
const MnvSmallCost kSmallGather{0.0992, 2.8, 2.0, 0.0}, kSmallFilter{0.1824, 4.3, 1.4, 3.9};
int small_gather_ranges(long long rows, int n, int small_slabs, int tile, long long tile_rows, int slabs, double fixed, size_t ws_floats,
                        double share = 1.0);
// where their vectors' offsets (channel planes, rows past the last) stay within 32 bits
bool small_reach(const ConvGeom& g) {
  const long long lim = (1LL << 28) - 1;
  return (long long)g.N * g.C * g.HW <= lim && (long long)g.N * g.K * g.HoWo <= lim && (long long)g.K * g.CRS <= lim;
}

int make_geom(ConvGeom* g, int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh,
              int R, int S) {
  if (N <= 0 || C <= 0 || K <= 0 || H <= 0 || W <= 0 || ph < 0 || pw < 0 || sv <= 0 ||
      sh <= 0 || R <= 0 || S <= 0)
    return MNV_ERR_INVALID;
  int Ho = (H + 2 * ph - R) / sv + 1, Wo = (W + 2 * pw - S) / sh + 1;
  if (H + 2 * ph < R || W + 2 * pw < S || Ho <= 0 || Wo <= 0) return MNV_ERR_INVALID;
  // 16-bit packed coordinates and 32-bit element offsets
  if (H + ph + R >= 16000 || W + pw + S >= 16000) return MNV_ERR_INVALID;
  const long long lim = (1LL << 29) - 1;  // 32-bit byte offsets into each tensor
  if ((long long)N * C * H * W > lim || (long long)N * K * Ho * Wo > lim ||
      (long long)K * C * R * S > lim)
    return MNV_ERR_INVALID;
  g->N = N; g->C = C; g->K = K; g->H = H; g->W = W; g->Ho = Ho; g->Wo = Wo;
  g->R = R; g->S = S; g->ph = ph; g->pw = pw; g->sv = sv; g->sh = sh;
  g->HW = H * W; g->HoWo = Ho * Wo; g->RS = R * S; g->CRS = C * R * S;
  g->d_RS = mnv_fastdiv_make(g->RS);
  g->d_S = mnv_fastdiv_make(S);
  g->d_HoWo = mnv_fastdiv_make(g->HoWo);
  g->d_Wo = mnv_fastdiv_make(Wo);
  g->d_HW = mnv_fastdiv_make(g->HW);
  g->d_W = mnv_fastdiv_make(W);
  g->d_sv = mnv_fastdiv_make(sv);
  g->d_sh = mnv_fastdiv_make(sh);
  return MNV_OK;
}

// Images per launch: bottom, top and filter are read through 32-bit byte offsets, so one
// launch takes at most 2^29 - 1 elements of each.  A larger batch (up to the reference's
// limit of 2^31 - 1 elements per tensor) runs as several launches over chunks of images --
// images are the slowest dimension, so a chunk is a contiguous slice of bottom and top --
// with the filter gradient accumulated chunk by chunk.  0: a single image (or the filter)
// is too large.
int images_per_launch(int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R, int S) {
  if (N <= 0 || C <= 0 || K <= 0 || H <= 0 || W <= 0 || ph < 0 || pw < 0 || sv <= 0 || sh <= 0 ||
      R <= 0 || S <= 0 || H + 2 * ph < R || W + 2 * pw < S)
    return 0;
  const long long lim = (1LL << 29) - 1;
  const long long Ho = (H + 2 * ph - R) / sv + 1, Wo = (W + 2 * pw - S) / sh + 1;
  const long long per_bottom = (long long)C * H * W, per_top = (long long)K * Ho * Wo;
  if ((long long)K * C * R * S > lim || per_bottom > lim || per_top > lim) return 0;
  if (per_bottom * N > 0x7fffffffLL || per_top * N > 0x7fffffffLL) return 0;
  long long chunk = lim / (per_bottom > per_top ? per_bottom : per_top);
  return (int)(chunk < N ? chunk : N);
}

int pick_tile(int m, int n) {
  if (n <= 32) return 3;
  long long big = (long long)((m + 127) / 128) * ((n + 127) / 128);
  if (big < 128 || m <= 64 || n <= 64) return 0;
  return wide_tile(n);
}

// A 64x64 or 128x32 tile does little arithmetic per k-slab, so a slab costs one trip to
// memory and back; its kernels need about 64 registers and at most 24 KB of LDS, which
// lets a CU hold six to eight workgroups whose trips overlap.  When the output has fewer tiles than that, the
// reduction is cut into k ranges (at least six slabs each) until about eight workgroups per
// CU are in flight.  `ws_floats`: workspace left for the partial results.
int small_tile_splits(int tile, int m, int n, int slabs, size_t ws_floats) {
  if (tile != 0 && tile != 3) return 1;
  const int bm = kTileM[tile], bn = kTileN[tile];
  long long tiles = (long long)((m + bm - 1) / bm) * ((n + bn - 1) / bn);
  const long long cus = mnv_cu_count();
  if (tiles >= 6 * cus) return 1;
  long long want = (8 * cus + tiles - 1) / tiles;
  if (want > slabs / 6) want = slabs / 6;
  size_t fit = ws_floats / ((size_t)m * n);
  if ((size_t)want > fit) want = (long long)fit;
  return want < 2 ? 1 : (int)want;
}

int small_gather_ranges(long long rows, int n, int small_slabs, int tile, long long tile_rows, int slabs, double fixed, size_t ws_floats,
                        double share) {
  if ((tile != 0 && tile != 3) || tile_rows > 0x7fffffff) return 0;
  const int splits = small_tile_splits(tile, (int)tile_rows, n, slabs, (size_t)-1);
  const long long tiles = (tile_rows + kTileM[tile] - 1) / kTileM[tile] * ((n + kTileN[tile] - 1) / kTileN[tile]);
  const double slab = (tile == 0 ? 0.28 : 0.46) * (double)tiles * splits / mnv_cu_count();
  double against = fixed + (slab > 0.3 ? slab : 0.3) * ((slabs + splits - 1) / splits);
  if (splits > 1) against += (tile == 0 ? 2.6 : 3.0) + (tile == 0 ? 1.6 : 0.7) * 8.0 * (double)tile_rows * n * splits / 6e6;
  return mnv_small_ranges(rows, n, small_slabs, ws_floats, kSmallGather, share * against);
}

// Workspace layout of the forward and data-gradient convolutions: the permuted filter
// (when the fast policy applies) first, then, 256-byte aligned, the partial results.
size_t align256(size_t bytes) { return (bytes + 255) & ~(size_t)255; }

// The reduction's channel count as the FAST policies take it, a multiple of 16, or 0 where the
// generic ones are to be used; `others` x RS x channels is the permuted filter, `rows` those of the product.
// Data gradients unless said otherwise, us, generic -> padded.
// Padding pays where it adds up to 60% (64 x 28 x 28 under 3 x 3, 20 channels 35 -> 30, but 17 26 -> 29), within one
// slab up to 100% (8 channels 15.1 -> 14.3) while the outputs are at most 32.  On 128 and more of the 64 x 64 tiles that
// more outputs take it may add 40%, in bf16 parts 60% (10 channels to 200, 16 x 28 x 28 under 3 x 3 25.3 -> 16.5,
// under 5 x 5 51.6 -> 28.7, but without parts on 16 x 14 x 14 20.8 -> 22.5; 8 to 40 on 16 x 28 x 28 17.2 -> 21.0; forward 8 to 128 on
// 64 x 28 x 28 46.7 -> 64.8, and in a few sizes that fill one round of the CUs the other way: 8 to 104 on 32 x 28 x 28 43 -> 29).
// Few tiles wait for one slab after the other, 1.5 us for a generic one and 0.65 for a padded one, which has to
// repay the launch that permutes the filter too (to 12 channels, 1 to 16 images of 14 x 14 or 28 x 28: under 1 x 1 from 8, 1
// slab each, 5.2 -> 6.4; from 24, 2, 6.8 -> 6.8; from 40, 3, 8.3 -> 7.5; under 3 x 3 from 8, 5 and 9, 11.2 -> 11.7; from 12, 7 and 9,
// 14.4 -> 12.2).  With tiles to fill the chip, two per CU, a single slab still does not, two do (24 to 312 on 50 x 23 x 14
// 24 -> 19).
int fast_channels(int channels, int others, int RS, long long rows) {
  const int width = (channels + 15) / 16 * 16;
  if (width != channels) {
    const long long tiles = (rows + 63) / 64 * ((others + 63) / 64);
    const long long slabs = ((long long)channels * RS + 15) / 16, padded = (long long)RS * (width / 16);
    const bool wide = others > 32;
    if (width > 16 ? 5 * width > 8 * channels : channels < 8) return 0;
    if (width == 16 && wide && tiles >= 128 && 5 * padded > 7 * slabs &&
        (5 * padded > 8 * slabs || !split_ranges((int)rows, others, (int)padded, pick_tile((int)rows, others), (size_t)-1)))
      return 0;
    if (tiles < 512 ? 7 * slabs <= 3 * padded + (wide ? 15 : 10) : slabs < 2) return 0;
  }
  return (long long)others * RS * width <= (1LL << 29) - 1 ? width : 0;
}
// the no-padding policy reads the filter where it is; for a small problem the extra launch that
// permutes the filter for the fast policy would cost more than it gains
bool unpadded_table(const ConvGeom& g) { return g.ph == 0 && g.pw == 0 && g.CRS <= 4096; }
// Forward, channels padded: only in bf16 parts, the generic gathers are as fast on the fp32
// instruction.  200 -> 200 channels under 3 x 3 on 16 x 14 x 14 61 -> 34 us, 64 x 28 x 28 470 -> 380, under 5 x 5 on
// 16 x 28 x 28 629 -> 214; without parts 24 -> 24 on 64 x 28 x 28 31 -> 33, 8 -> 8 10 -> 15.
int fwd_channels(const ConvGeom& g) {
  const int m = g.N * g.HoWo, tile = pick_tile(m, g.K);
  const bool off = g.C % 16 != 0;
  if (unpadded_table(g) && (tile == 0 || tile == 3 || off)) return 0;
  const int width = fast_channels(g.C, g.K, g.RS, m);
  return off && width && !split_ranges(m, g.K, g.RS * (width / 16), tile, (size_t)-1) ? 0 : width;
}
// Up to four slabs and more than three small tiles per CU: their first loads and last stores are what counts, and larger tiles have
// fewer.  Under 1 x 1, 24 -> 96 on 15 x 22 x 43 7.7 -> 9.1 us, 24 -> 32 on 78 x 9 x 56 6.6 -> 8.7, 32 -> 176 on 5 x 48 x 29 7.3 -> 8.3, data
// gradient 176 <- 56 on 10 x 10 x 45 8.6 -> 9.6; 64 -> 168 on 26 x 9 x 11 (1.9 tiles) 7.3 -> 5.7.  Of 25 random layers 16 lost, two gained
// more than 6% (360 <- 56 on 3 x 23 x 51 15.6 -> 12.2).
bool small_stores_bound(long long m, int n, int slabs) {
  return slabs <= 4 && (m + MNV_SMALL_TILE - 1) / MNV_SMALL_TILE * ((n + MNV_SMALL_TILE - 1) / MNV_SMALL_TILE) > 3LL * mnv_cu_count();
}
// The forward pass on the small tiles: their k ranges (0: not), and the channels of the permuted filter
// (0: the filter as it is).  From 16 channels on the generic gathers of padded layers are left for the permuted filter, unless
// permuting it costs more: 6 us per million values beyond those that the estimate was fitted to (5 x 5 at stride 2, 200 -> 328 on 4 x 10 x 8
// 14.3 -> 20.1 us, 264 -> 264 on 6 x 19 x 8 31.4 -> 36.1, 104 -> 384 on 2 x 11 x 25 17.2 -> 19.1).
struct SmallForward {
  int z = 0, width = 0;
  size_t filter_bytes = 0;
};
SmallForward small_forward(const ConvGeom& g, size_t ws_bytes) {
  SmallForward p;
  const int m = g.N * g.HoWo, tile = pick_tile(m, g.K), width = fwd_channels(g);
  if (!small_reach(g)) return p;
  const int slabs = width ? g.RS * (width / 16) : (g.CRS + 15) / 16;
  if ((width || unpadded_table(g)) && split_ranges(m, g.K, slabs, tile, (size_t)-1)) return p;
  p.width = width || unpadded_table(g) || g.C < 16 ? width : fast_channels(g.C, g.K, g.RS, m);
  if (!p.width && !unpadded_table(g)) return p;
  p.filter_bytes = (size_t)g.K * g.RS * p.width * sizeof(float);
  if (p.filter_bytes > ws_bytes) return p;
  const size_t left = ws_bytes > align256(p.filter_bytes) ? (ws_bytes - align256(p.filter_bytes)) / sizeof(float) : 0;
  const int own = p.width ? g.RS * (p.width / 16) : slabs;
  if (small_stores_bound(m, g.K, own)) return p;
  const double permute = p.width && !width ? std::max(0.0, 6e-6 * ((double)g.K * g.RS * p.width - 4e5)) : 0.0;
  // Strides above 1 scatter the positions that a load gathers, and a slab of the small tiles takes longer than its estimate.  Without
  // padding they gain below 80% of the other launch's (336 random layers, 0.82 of the time), above
  // they do not (45, 1.02; 216 -> 24 under 5 x 5 on 35 x 34 x 8 22.2 -> 40.7 us); padded layers still do (47, 0.94).
  p.z = small_gather_ranges(m, g.K, own, tile, m, slabs, 1.0 - permute, left, !g.ph && !g.pw && (g.sv > 1 || g.sh > 1) ? 0.92 : 1.0);
  return p;
}
size_t small_bytes(size_t filter_bytes, int z, size_t results) {
  return z > 1 ? align256(filter_bytes) + z * results * sizeof(float) : filter_bytes;
}
// Data gradient: the generic gathers also divide by the strides and lose wherever padding pays.  200 <- 200
// channels under 3 x 3 on 16 x 14 x 14 65 -> 34 us, 64 x 28 x 28 612 -> 375, under 5 x 5 on 16 x 28 x 28 838 -> 216;
// 40 <- 40 on 16 x 14 x 14 16.2 -> 13.7.
int bwd_data_channels(const ConvGeom& g) {
  return g.sv == 1 && g.sh == 1 ? fast_channels(g.K, g.C, g.RS, (long long)g.N * g.HW) : 0;
}

// The data gradient of strides above 1, phase by phase (ConvBwdDataPhases).  us, generic gathers -> phases, at stride 2: 344 <- 112 channels under
// 5 x 5 on 104 x 15 x 45 1780 -> 249, 264 <- 216 on 45 x 33 x 38 2293 -> 453, 128 <- 128 under 1 x 1 on 88 x 15 x 20 32 -> 31, 320 <- 96
// under 3 x 3 on 41 x 14 x 29 191 -> 64, 48 <- 184 on 17 x 16 x 15 26.6 -> 19.1.  Few tiles of few slabs are bound by one
// trip to memory after the other, 1.45 us for a generic slab and 0.65 for one of a phase, and pay for the launch that permutes the filter,
// 5.5 us in all: 11 channels under 1 x 1 5.0 -> 10.2, 70 10.3 -> 10.9, 16 under 3 x 3 15.1 -> 9.7.  Many tiles are bound by their
// stores, which leave every sh-th float (about 1 TB/s, and 20 us before the first slab counts), and repay them from five generic slabs
// on, and nine of a CU's 128 x 128 tiles: under 1 x 1, 256 <- 32 on 52 x 14 x 12 14.8 -> 29.2, 328 <- 32 on 93 x 53 x 22 73 -> 121, 224 <- 128
// on 69 x 32 x 7 30.1 -> 37.9 (all left to the generic gathers), 192 <- 72 on 39 x 21 x 54 36 -> 28, 208 <- 128 on 26 x 50 x 45 73 -> 47.  600
// random layers at stride 2: by taking all of two slabs on, 38 lost more than 3%, up to 2 times; by this rule 2, up to 1.18; the dearest win that
// it leaves is 216 <- 104 on 36 x 17 x 34, 42 -> 35.  Error against float64 (525 random layers): 0.74 of that of
// the generic gathers, 0.37 where they run in parts; 26 above 1.02 times, by up to 1.05 on large tiles and 1.15 on small ones.  Without the rules
// below for parts and small tiles 37 of the large and 23 of the small ones were, by up to 1.36 and 2.1, for up to 1.5 times less time: 48 <- 24
// under 3 x 3 on 120 x 27 x 30 1.47e-7 -> 0.81e-7 (generic 1.08e-7), 29 -> 43 us (70); 112 <- 48 on 51 x 33 x 50 2.05e-7 -> 0.66e-7 (1.91e-7), 51 -> 67 (143).
struct PhasePlan {
  int width = 0;  // channels as the policy takes them; 0: the generic gathers
  int tile = 0, parts = 0, splits = 1, phase_rows = 0, slabs = 0;  // parts > 0: bf16 parts with that many k ranges
  bool small = false;  // the small tiles with `splits`
  size_t filter_bytes = 0, rows = 0;
  size_t partial_bytes(int n) const { return parts > 1 || splits > 1 ? (size_t)(parts ? parts : splits) * rows * n * sizeof(float) : 0; }
};
// Classes of a dimension's positions modulo the stride that hold one.
long long phase_classes(int stride, int extent) { return stride < extent ? stride : extent; }
PhasePlan phase_plan(const ConvGeom& g, size_t ws_bytes) {
  PhasePlan p;
  if (g.sv == 1 && g.sh == 1) return p;
  const int width = (g.K + 15) / 16 * 16, spp = width / 16;
  const long long phases = phase_classes(g.sv, g.H) * phase_classes(g.sh, g.W);
  const long long most = (long long)g.N * ((g.H - 1) / g.sv + 1) * ((g.W - 1) / g.sh + 1);  // rows of a phase
  p.filter_bytes = (size_t)g.C * g.RS * width * sizeof(float);
  if ((long long)g.C * g.RS * width > (1LL << 29) - 1 || ws_bytes < p.filter_bytes) return p;
  // rows of all phases on the tallest tile: within an int, for tiny phases by the million are not
  if (phases > 0x3fffffff / ((most + 127) / 128 * 128)) return p;
  const size_t left = ws_bytes > align256(p.filter_bytes) ? (ws_bytes - align256(p.filter_bytes)) / sizeof(float) : 0;
  // what the launch shapes are chosen by: a product of all positions and the mean extent of k
  p.slabs = ((g.R - 1) / g.sv + 1) * ((g.S - 1) / g.sh + 1) * spp;
  const int m = g.N * g.HW, mean = (int)std::min<long long>(((long long)g.RS * spp + phases - 1) / phases, p.slabs);
  p.tile = pick_tile(m, g.C);
  auto rows_on = [&](int tile_rows) {
    p.phase_rows = (int)((most + tile_rows - 1) / tile_rows * tile_rows);
    p.rows = (size_t)p.phase_rows * phases;
  };
  // No sum is to be longer than that of the generic gathers, which cut the tail of their large tiles, and the k of their small ones,
  // into more ranges: where they shorten more than a tenth of the sums by a tail (5% of the error) the phases run in parts, and where they have
  // more ranges, on the small tiles, which sum in runs.
  const int generic_slabs = (int)(((long long)g.K * g.RS + 15) / 16);
  rows_on(128);
  p.parts = split_ranges(m, g.C, mean, p.tile, left / (p.rows ? p.rows : 1) * m);
  if (!p.parts && (p.tile == 1 || p.tile == 2)) {
    const long long tiles = (m + 127LL) / 128 * ((g.C + kTileN[p.tile] - 1) / kTileN[p.tile]);
    const MnvTailPlan t = mnv_tail_plan(tiles, generic_slabs, (size_t)kTileM[p.tile] * kTileN[p.tile], (size_t)-1 / sizeof(float));
    if (t.z > 1 && (double)(tiles - t.begin) / tiles * (1.0 - 1.0 / t.z) > 0.1) p.parts = 1;
  }
  if (!p.parts) {
    rows_on(kTileM[p.tile]);
    p.splits = small_tile_splits(p.tile, (int)p.rows, g.C, p.slabs, left);
    const long long tile_rows = (long long)p.rows;
    rows_on(MNV_SMALL_TILE);
    int z = 0;
    if (small_reach(g) && (p.tile == 0 || p.tile == 3)) {
      z = small_gather_ranges((long long)p.rows, g.C, mean, p.tile, tile_rows, mean, 2.0, left);
      if (!z && small_tile_splits(p.tile, m, g.C, generic_slabs, (size_t)-1) > p.splits)
        z = mnv_small_ranges((long long)p.rows, g.C, mean, left, kSmallGather, 1e30);
    }
    if (z) {
      p.small = true;
      p.splits = z;
    } else {
      rows_on(kTileM[p.tile]);
    }
  }
  // the tiles' rows, and channels, are filled up: not where that multiplies more than the generic gathers
  if ((long long)p.rows * width >= (long long)m * g.K * phases) return p;
  const long long tiles = (m + 63LL) / 64 * ((g.C + 63) / 64), slabs = ((long long)g.K * g.RS + 15) / 16;
  const long long cus = mnv_cu_count(), big = std::max((m + 127LL) / 128 * ((g.C + 127) / 128), cus);
  if (tiles < 512 ? 11 * slabs <= 5 * p.slabs + 42 : slabs < 5 || slabs * big <= 9 * cus) return p;
  p.width = width;
  return p;
}

// The data gradient of unit strides on the small tiles: their k ranges, 0: not.
int small_bwd_data(const ConvGeom& g, int width, size_t ws_bytes) {
  const size_t filter_bytes = (size_t)g.C * g.RS * width * sizeof(float);
  if (!width || filter_bytes > ws_bytes || !small_reach(g)) return 0;
  const int m = g.N * g.HW, tile = pick_tile(m, g.C), slabs = g.RS * (width / 16);
  if (split_ranges(m, g.C, slabs, tile, (size_t)-1)) return 0;
  const size_t left = ws_bytes > align256(filter_bytes) ? (ws_bytes - align256(filter_bytes)) / sizeof(float) : 0;
  return small_stores_bound(m, g.C, slabs) ? 0 : small_gather_ranges(m, g.C, slabs, tile, m, slabs, 2.0, left);
}

// k ranges of the filter gradient: up to 256, and up to 512 for outputs of at most 16384
// elements, whose partial results cost next to nothing (the MNIST CNN's filters: its step
// 0.28 -> 0.25 ms; conv1 of the AlexNet shape with 341 ranges instead of 255: 0.50 -> 0.54 ms).
#define MNV_BWDF_MAX_SPLITS 256
#define MNV_BWDF_MAX_SPLITS_SMALL 512

// The filter gradient gets its parallelism from splitting the long N*Ho*Wo reduction,
// so it keeps the 128x128 tile (twice the operand reuse) unless the output is tiny.
int bwd_filter_tile(int m, int n) {
  if (n <= 32) return 3;
  return (m <= 64 || n <= 64) ? 0 : wide_tile(n);
}

int bwd_filter_splits(int m, int n, int k, size_t ws_floats, double* cost = nullptr) {
  const int tile = bwd_filter_tile(m, n);
  const int bm = kTileM[tile], bn = kTileN[tile];
  long long tiles = (long long)((m + bm - 1) / bm) * ((n + bn - 1) / bn);
  int slabs = (k + 15) / 16;
  int max_splits = (size_t)m * n <= 16384 ? MNV_BWDF_MAX_SPLITS_SMALL : MNV_BWDF_MAX_SPLITS;
  if (max_splits > slabs / 8) max_splits = slabs / 8;
  size_t fit = ws_floats / ((size_t)m * n);
  if ((size_t)max_splits > fit) max_splits = (int)fit;
  return mnv_pick_splits(tiles, slabs, max_splits, mnv_cu_count(), 0.0, cost);
}

// The filter gradient on the small tiles instead of k ranges of the others: their number, 0: not; `slabs` as the policies with a
// table of positions count them.  In us, an estimate of mnv_pick_splits is worth 0.47, 0.74, 0.51 and 0.39 on the four tiles, beside 1.3,
// 2.6, 4.5 and 3.6 and the partial results at 3.3, 3.9, 3 and 5.6 TB/s (10% off, rms, on 194 layers).
// us: 352 <- 48 channels under 3 x 3, stride 2, on 2 x 27 x 36 22.8 -> 11.0, 344 <- 40 under 5 x 5 on 43 x 13 25 -> 10,
// 64 <- 288 on 7 x 26 x 19 48 -> 36.
int small_filter_ranges(const ConvGeom& g, int slabs, size_t ws_floats) {
  static const double fixed[4] = {1.3, 2.6, 4.5, 3.6}, unit[4] = {0.468, 0.738, 0.507, 0.385}, bytes[4] = {1.83, 1.55, 1.98, 1.07};
  if (!small_reach(g)) return 0;
  double cost;
  const int tile = bwd_filter_tile(g.CRS, g.K), z = bwd_filter_splits(g.CRS, g.K, g.N * g.HoWo, (size_t)-1, &cost);
  const double against = fixed[tile] + unit[tile] * cost + (z > 1 ? bytes[tile] * 8.0 * (double)g.CRS * g.K * z / 6e6 : 0.0);
  return mnv_small_ranges(g.CRS, g.K, slabs, ws_floats, kSmallFilter, against);
}
// Positions of an image, as those policies pad them, and whether the table of `taps` taps fits beside the tiles.
int filter_positions(const ConvGeom& g) { return (g.HoWo + 15) / 16 * 16; }
bool filter_table(const ConvGeom& g, int taps) { return (size_t)taps * filter_positions(g) * 4 <= 24 * 1024; }
// Taps whose rows, in (tap, channel) order, meet one tile of `rows`, over all tiles: 1 when `rows` divides
// C, never more than (rows + C - 1) / C + 1.
int filter_taps(const ConvGeom& g, int rows) {
  int taps = 1;
  for (int m0 = 0; m0 < g.CRS; m0 += rows) {
    const int last = (m0 + rows - 1 < g.CRS ? m0 + rows - 1 : g.CRS - 1) / g.C;
    if (last - m0 / g.C + 1 > taps) taps = last - m0 / g.C + 1;
    if (m0 / rows >= g.C) break;  // the pattern of m0 % C repeats after C tiles
  }
  return taps;
}

}  // namespace

extern "C" {

size_t mnv_conv_fwd_workspace_bytes(int N, int C, int K, int H, int W, int ph, int pw, int sv,
                                   int sh, int R, int S) {
  ConvGeom g;
  if (make_geom(&g, N, C, K, H, W, ph, pw, sv, sh, R, S)) return 0;
  const SmallForward small = small_forward(g, (size_t)-1);
  const bool wino = mnv_wino_images(N, C, K, H, W, ph, pw, R, S, sv, sh, (size_t)-1);
  if (small.z && !wino) return small_bytes(small.filter_bytes, small.z, (size_t)N * g.HoWo * K);
  const int width = fwd_channels(g);
  const size_t permuted = (size_t)K * g.RS * width * sizeof(float);
  const int gm = N * g.HoWo, gn = K, slabs = width ? g.RS * (width / 16) : (g.CRS + 15) / 16;
  const int splits = small_tile_splits(pick_tile(gm, gn), gm, gn, slabs, (size_t)-1);
  const size_t tail = tail_workspace_bytes(pick_tile(gm, gn), gm, gn, slabs, width || unpadded_table(g));
  size_t need = tail ? align256(permuted) + tail
                     : splits > 1 ? align256(permuted) + (size_t)splits * gm * gn * sizeof(float) : permuted;
  const size_t parts = split_bytes(pick_tile(gm, gn), gm, gn, slabs);
  if (parts && align256(permuted) + parts > need) need = align256(permuted) + parts;
  if (wino) {
    const size_t w = mnv_wino_workspace_bytes(N, C, K, H, W, ph, pw, R);
    if (w > need) need = w;
  }
  return need;
}

static int conv_fwd_impl(const float* bottom, const float* filter, const float* bias, float* top,
                         int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R,
                         int S, void* workspace, size_t workspace_bytes, mnv_stream_t stream,
                         int relu, DirectPlan* report_to = nullptr) {
  ConvGeom g;
  if (!report_to && (!bottom || !filter || !bias || !top)) return MNV_ERR_INVALID;
  int rc = make_geom(&g, N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (rc) return rc;
  int gm = N * g.HoWo, gn = K, gk = g.CRS;
  hipStream_t s = mnv_stream(stream);
  // 3 x 3 and 5 x 5 unit-stride layers with enough channels and tiles: minimal filtering, see
  // winograd.hip (its transformed tensors are read and written in 16-byte vectors)
  if (const int images = mnv_wino_images(N, C, K, H, W, ph, pw, R, S, sv, sh,
                                         workspace && mnv_aligned16(workspace) ? workspace_bytes : 0))
    return report_to ? report(report_to, 0, 1, 1)
                     : mnv_wino_conv(bottom, filter, bias, nullptr, top, N, C, K, H, W, ph, pw, R, 0, relu, images,
                                     workspace, workspace_bytes, s);
  if (const SmallForward small = small_forward(g, workspace ? workspace_bytes : 0); small.z) {
    if (report_to) return report(report_to, MNV_SMALL_TILE, small.z, 0);
    float* wp = static_cast<float*>(workspace);
    float* part = small.z > 1 ? reinterpret_cast<float*>(static_cast<char*>(workspace) + align256(small.filter_bytes)) : nullptr;
    if (!small.width)
      return mnv_gemm_small_launch(ConvFwdNP{bottom, filter, bias, top, g, gm, gn, gk, (gk + 15) / 16, gk >= 16 ? gk / 16 : 1, relu},
                                   small.z, part, s);
    rc = permute_filter(filter, wp, K, C, R, S, small.width, false, s);
    if (rc) return rc;
    const int spp = small.width / 16;
    if (small.width != C)
      return mnv_gemm_small_launch(ConvOneRow<ConvFwd<true, true>, true>{{bottom, wp, bias, top, g, gm, gn, gk, g.RS * spp, spp, relu}},
                                   small.z, part, s);
    return mnv_gemm_small_launch(ConvOneRow<ConvFwd<true>, false>{{bottom, wp, bias, top, g, gm, gn, gk, g.RS * spp, spp, relu}},
                                 small.z, part, s);
  }
  const int tile = pick_tile(gm, gn);
  int width = fwd_channels(g);
  const size_t permuted_bytes = (size_t)K * g.RS * width * sizeof(float);
  const bool np = unpadded_table(g);
  if (!workspace || workspace_bytes < permuted_bytes) width = 0;
  const bool fast = width != 0;
  // what is left of the workspace after the permuted filter holds the partial results
  const size_t used = fast ? align256(permuted_bytes) : 0;
  float* part = workspace && workspace_bytes > used ? reinterpret_cast<float*>(static_cast<char*>(workspace) + used) : nullptr;
  const int splits = small_tile_splits(tile, gm, gn, fast ? g.RS * (width / 16) : (gk + 15) / 16,
                                       part ? (workspace_bytes - used) / sizeof(float) : 0);
  if (fast) {
    float* wp = static_cast<float*>(workspace);
    rc = report_to ? MNV_OK : permute_filter(filter, wp, K, C, R, S, width, false, s);
    if (rc) return rc;
    const int spp = width / 16;
    const size_t part_bytes = part ? workspace_bytes - used : 0;
    if (width != C)
      return launch_direct(tile, ConvFwd<true, true>{bottom, wp, bias, top, g, gm, gn, gk, g.RS * spp, spp, relu}, splits,
                           part, s, part_bytes, report_to);
    return launch_direct(tile, ConvFwd<true>{bottom, wp, bias, top, g, gm, gn, gk, g.RS * spp, spp, relu}, splits, part, s,
                         part_bytes, report_to);
  }
  if (np) {
    ConvFwdNP p{bottom, filter, bias, top, g, gm, gn, gk, (gk + 15) / 16, gk >= 16 ? gk / 16 : 1, relu};
    // four taps of a filter row at a time where its rows divide so
    const size_t part_bytes = part ? workspace_bytes - used : 0;
    const int z = split_ranges(gm, gn, p.total_slabs, tile, part_bytes / sizeof(float));
    if (z && ConvFwdRows::takes(S)) {
      ConvFwdRows q{};
      static_cast<ConvFwdNP&>(q) = p;
      q.per_row = (S + 3) / 4;
      q.groups = C * R * q.per_row;
      q.K = 4 * q.groups;
      q.total_slabs = q.spp = (q.groups + 3) / 4;
      q.d_per_row = mnv_fastdiv_make(q.per_row);
      q.d_R = mnv_fastdiv_make(R);
      return launch_parts(q, z, part, s, part_bytes, report_to);
    }
    return launch_direct(tile, p, splits, part, s, part ? workspace_bytes - used : 0, report_to);
  }
  ConvFwd<false> p{bottom, filter, bias, top, g, gm, gn, gk, (gk + 15) / 16, 1, relu};
  return launch_tile(tile, p, splits, part, s, part ? workspace_bytes - used : 0, report_to);
}

static int conv_fwd_chunks(const float* bottom, const float* filter, const float* bias, float* top,
                           int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R,
                           int S, void* workspace, size_t workspace_bytes, mnv_stream_t stream,
                           int relu) {
  const int chunk = images_per_launch(N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (chunk <= 0 || chunk >= N)  // the usual case, and invalid geometry (refused inside)
    return conv_fwd_impl(bottom, filter, bias, top, N, C, K, H, W, ph, pw, sv, sh, R, S, workspace,
                         workspace_bytes, stream, relu);
  if (!bottom || !top) return MNV_ERR_INVALID;
  const size_t per_bottom = (size_t)C * H * W;
  const size_t per_top = (size_t)K * ((H + 2 * ph - R) / sv + 1) * ((W + 2 * pw - S) / sh + 1);
  for (int n0 = 0; n0 < N; n0 += chunk) {
    const int nn = N - n0 < chunk ? N - n0 : chunk;
    int rc = conv_fwd_impl(bottom + n0 * per_bottom, filter, bias, top + n0 * per_top, nn, C, K, H,
                           W, ph, pw, sv, sh, R, S, workspace, workspace_bytes, stream, relu);
    if (rc) return rc;
  }
  return MNV_OK;
}

int mnv_conv_fwd(const float* bottom, const float* filter, const float* bias, float* top, int N,
                 int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R, int S,
                 void* workspace, size_t workspace_bytes, mnv_stream_t stream) {
  return conv_fwd_chunks(bottom, filter, bias, top, N, C, K, H, W, ph, pw, sv, sh, R, S, workspace,
                         workspace_bytes, stream, 0);
}

int mnv_conv_fwd_relu(const float* bottom, const float* filter, const float* bias, float* top,
                      int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R,
                      int S, void* workspace, size_t workspace_bytes, mnv_stream_t stream) {
  return conv_fwd_chunks(bottom, filter, bias, top, N, C, K, H, W, ph, pw, sv, sh, R, S, workspace,
                         workspace_bytes, stream, 1);
}

size_t mnv_conv_bwd_data_workspace_bytes(int N, int C, int K, int H, int W, int ph, int pw,
                                        int sv, int sh, int R, int S) {
  ConvGeom g;
  if (make_geom(&g, N, C, K, H, W, ph, pw, sv, sh, R, S)) return 0;
  const PhasePlan phases = phase_plan(g, (size_t)-1);
  if (phases.width) {
    const size_t partial = phases.partial_bytes(C);
    return partial ? align256(phases.filter_bytes) + partial : phases.filter_bytes;
  }
  const int width = bwd_data_channels(g);
  const size_t permuted = (size_t)C * g.RS * width * sizeof(float);
  const bool wino = mnv_wino_images(N, K, C, g.Ho, g.Wo, R - 1 - ph, S - 1 - pw, R, S, sv, sh, (size_t)-1);
  if (const int z = wino ? 0 : small_bwd_data(g, width, (size_t)-1)) return small_bytes(permuted, z, (size_t)N * g.HW * C);
  const int gm = N * g.HW, gn = C, slabs = width ? g.RS * (width / 16) : (K * g.RS + 15) / 16;
  const int splits = small_tile_splits(pick_tile(gm, gn), gm, gn, slabs, (size_t)-1);
  const size_t tail = tail_workspace_bytes(pick_tile(gm, gn), gm, gn, slabs, width);
  size_t need = tail ? align256(permuted) + tail
                     : splits > 1 ? align256(permuted) + (size_t)splits * gm * gn * sizeof(float) : permuted;
  const size_t parts = split_bytes(pick_tile(gm, gn), gm, gn, slabs);
  if (parts && align256(permuted) + parts > need) need = align256(permuted) + parts;
  if (wino) {
    const size_t w = mnv_wino_workspace_bytes(N, K, C, g.Ho, g.Wo, R - 1 - ph, S - 1 - pw, R);
    if (w > need) need = w;
  }
  return need;
}

static int bwd_data_phases(const float* top_diff, const float* filter, const float* gate, float* bottom_diff, const ConvGeom& g,
                           const PhasePlan& plan, void* workspace, hipStream_t s) {
  float* permuted = static_cast<float*>(workspace);
  float* part = plan.partial_bytes(g.C) ? reinterpret_cast<float*>(static_cast<char*>(workspace) + align256(plan.filter_bytes)) : nullptr;
  const int rc = permute_filter(filter, permuted, g.K, g.C, g.R, g.S, plan.width, true, s, g.sv, g.sh);
  if (rc) return rc;
  auto launch = [&](auto p) {
    p.top_diff = top_diff; p.filter = permuted; p.bottom_diff = bottom_diff; p.gate = gate;
    p.g = g;
    p.M = (int)plan.rows; p.N = g.C; p.total_slabs = plan.slabs; p.spp = plan.width / 16;
    p.phase_rows = plan.phase_rows;
    // class 0 holds the tap r' = 0, which meets output row i at input row i sv - ph + R - 1
    auto first = [](int reach, int stride, int* at, int* out) {
      *at = reach % stride < 0 ? reach % stride + stride : reach % stride;
      *out = (*at - reach) / stride;
    };
    first(g.R - 1 - g.ph, g.sv, &p.a0, &p.i00);
    first(g.S - 1 - g.pw, g.sh, &p.b0, &p.j00);
    p.hq = g.H / g.sv; p.hr = g.H % g.sv; p.wq = g.W / g.sh; p.wr = g.W % g.sh;
    p.rq = g.R / g.sv; p.rr = g.R % g.sv; p.sq = g.S / g.sh; p.sr = g.S % g.sh;
    p.col_classes = (int)phase_classes(g.sh, g.W);
    p.d_cols = mnv_fastdiv_make(p.col_classes);
    p.d_rows = mnv_fastdiv_make(p.phase_rows);
    for (int more = 0; more < 4; ++more) {
      const int plane = (p.hq + more / 2) * (p.wq + more % 2);  // 0: no position is in such a class
      p.d_plane[more] = mnv_fastdiv_make(plane ? plane : 1);
    }
    for (int more = 0; more < 2; ++more) {
      p.d_width[more] = mnv_fastdiv_make(p.wq + more ? p.wq + more : 1);
      p.d_taps[more] = mnv_fastdiv_make(p.sq + more ? p.sq + more : 1);
    }
    if (plan.small) {
      ConvOneRow<decltype(p), decltype(p)::PADDED> q;
      static_cast<decltype(p)&>(q) = p;
      return mnv_gemm_small_launch(q, plan.splits, part, s);
    }
    return plan.parts ? launch_parts(p, plan.parts, part, s, 0) : launch_tile(plan.tile, p, plan.splits, part, s);
  };
  return plan.width != g.K ? launch(ConvBwdDataPhases<true>{}) : launch(ConvBwdDataPhases<false>{});
}

static int conv_bwd_data_impl(const float* top_diff, const float* filter, const float* gate,
                              float* bottom_diff, int N, int C, int K, int H, int W, int ph,
                              int pw, int sv, int sh, int R, int S, void* workspace,
                              size_t workspace_bytes, mnv_stream_t stream, DirectPlan* report_to = nullptr) {
  ConvGeom g;
  if (!report_to && (!top_diff || !filter || !bottom_diff)) return MNV_ERR_INVALID;
  int rc = make_geom(&g, N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (rc) return rc;
  int gm = N * g.HW, gn = C, gk = K * g.RS;
  hipStream_t s = mnv_stream(stream);
  // the same correlation, of top_diff with the unflipped filters, under a padding of R - 1 - pad
  if (const int images = mnv_wino_images(N, K, C, g.Ho, g.Wo, R - 1 - ph, S - 1 - pw, R, S, sv, sh,
                                         workspace && mnv_aligned16(workspace) ? workspace_bytes : 0))
    return report_to ? report(report_to, 0, 1, 1)
                     : mnv_wino_conv(top_diff, filter, nullptr, gate, bottom_diff, N, K, C, g.Ho, g.Wo, R - 1 - ph,
                                     S - 1 - pw, R, 1, 0, images, workspace, workspace_bytes, s);
  if (sv > 1 || sh > 1) {
    const PhasePlan plan = phase_plan(g, workspace ? workspace_bytes : 0);
    if (plan.width && report_to) {
      report_to->classes = (int)(plan.rows / plan.phase_rows);
      return plan.parts ? report(report_to, 128, plan.parts, 1)
                        : report(report_to, plan.small ? MNV_SMALL_TILE : kTileM[plan.tile], plan.splits, 0);
    }
    if (plan.width) return bwd_data_phases(top_diff, filter, gate, bottom_diff, g, plan, workspace, s);
  }
  const int tile = pick_tile(gm, gn);
  const int width = bwd_data_channels(g);
  const size_t permuted_bytes = (size_t)C * g.RS * width * sizeof(float);
  const bool fast = width && workspace && workspace_bytes >= permuted_bytes;
  const size_t used = fast ? align256(permuted_bytes) : 0;
  float* part = workspace && workspace_bytes > used ? reinterpret_cast<float*>(static_cast<char*>(workspace) + used) : nullptr;
  const int splits = small_tile_splits(tile, gm, gn, fast ? g.RS * (width / 16) : (gk + 15) / 16,
                                       part ? (workspace_bytes - used) / sizeof(float) : 0);
  if (fast) {
    float* wq = static_cast<float*>(workspace);
    rc = report_to ? MNV_OK : permute_filter(filter, wq, K, C, R, S, width, true, s);
    if (rc) return rc;
    const int spp = width / 16;
    const size_t part_bytes = part ? workspace_bytes - used : 0;
    if (const int z = small_bwd_data(g, width, workspace_bytes)) {
      if (report_to) return report(report_to, MNV_SMALL_TILE, z, 0);
      if (width != K)
        return mnv_gemm_small_launch(ConvOneRow<ConvBwdData<true, true>, true>{{top_diff, wq, bottom_diff, g, gm, gn, gk, g.RS * spp, spp, gate}},
                                     z, part, s);
      return mnv_gemm_small_launch(ConvOneRow<ConvBwdData<true>, false>{{top_diff, wq, bottom_diff, g, gm, gn, gk, g.RS * spp, spp, gate}},
                                   z, part, s);
    }
    if (width != K)
      return launch_direct(tile, ConvBwdData<true, true>{top_diff, wq, bottom_diff, g, gm, gn, gk, g.RS * spp, spp, gate},
                           splits, part, s, part_bytes, report_to);
    return launch_direct(tile, ConvBwdData<true>{top_diff, wq, bottom_diff, g, gm, gn, gk, g.RS * spp, spp, gate}, splits,
                         part, s, part_bytes, report_to);
  }
  ConvBwdData<false> p{top_diff, filter, bottom_diff, g, gm, gn, gk, (gk + 15) / 16, 1, gate};
  return launch_tile(tile, p, splits, part, s, part ? workspace_bytes - used : 0, report_to);
}

static int conv_bwd_data_chunks(const float* top_diff, const float* filter, const float* gate,
                                float* bottom_diff, int N, int C, int K, int H, int W, int ph,
                                int pw, int sv, int sh, int R, int S, void* workspace,
                                size_t workspace_bytes, mnv_stream_t stream) {
  const int chunk = images_per_launch(N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (chunk <= 0 || chunk >= N)
    return conv_bwd_data_impl(top_diff, filter, gate, bottom_diff, N, C, K, H, W, ph, pw, sv, sh, R,
                              S, workspace, workspace_bytes, stream);
  if (!top_diff || !bottom_diff) return MNV_ERR_INVALID;
  const size_t per_bottom = (size_t)C * H * W;
  const size_t per_top = (size_t)K * ((H + 2 * ph - R) / sv + 1) * ((W + 2 * pw - S) / sh + 1);
  for (int n0 = 0; n0 < N; n0 += chunk) {
    const int nn = N - n0 < chunk ? N - n0 : chunk;
    int rc = conv_bwd_data_impl(top_diff + n0 * per_top, filter, gate ? gate + n0 * per_bottom : nullptr,
                                bottom_diff + n0 * per_bottom, nn, C, K, H, W, ph, pw, sv, sh, R, S,
                                workspace, workspace_bytes, stream);
    if (rc) return rc;
  }
  return MNV_OK;
}

int mnv_conv_bwd_data(const float* top_diff, const float* filter, float* bottom_diff, int N,
                      int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R, int S,
                      void* workspace, size_t workspace_bytes, mnv_stream_t stream) {
  return conv_bwd_data_chunks(top_diff, filter, nullptr, bottom_diff, N, C, K, H, W, ph, pw, sv, sh,
                              R, S, workspace, workspace_bytes, stream);
}

int mnv_conv_bwd_data_relu(const float* top_diff, const float* filter, const float* bottom,
                           float* bottom_diff, int N, int C, int K, int H, int W, int ph, int pw,
                           int sv, int sh, int R, int S, void* workspace, size_t workspace_bytes,
                           mnv_stream_t stream) {
  if (!bottom) return MNV_ERR_INVALID;
  return conv_bwd_data_chunks(top_diff, filter, bottom, bottom_diff, N, C, K, H, W, ph, pw, sv, sh,
                              R, S, workspace, workspace_bytes, stream);
}

size_t mnv_conv_bwd_filter_workspace_bytes(int N, int C, int K, int H, int W, int ph, int pw,
                                           int sv, int sh, int R, int S) {
  ConvGeom g;
  if (make_geom(&g, N, C, K, H, W, ph, pw, sv, sh, R, S)) return 0;
  int splits = bwd_filter_splits(g.CRS, K, N * g.HoWo, (size_t)-1);
  size_t bytes = splits > 1 ? (size_t)splits * g.CRS * K * sizeof(float) : 0;
  // the stream-k plan of the large tiles: at most four workgroups per CU, a partial tile each
  // and one more per output tile
  const int tile = bwd_filter_tile(g.CRS, K);
  if (tile == 1 || tile == 2) {
    const long long tiles = (long long)((g.CRS + kTileM[tile] - 1) / kTileM[tile]) *
                            ((K + kTileN[tile] - 1) / kTileN[tile]);
    const size_t sk = (size_t)(4 * mnv_cu_count() + tiles) * kTileM[tile] * kTileN[tile] * sizeof(float);
    if (tiles <= 4LL * mnv_cu_count() && sk > bytes) bytes = sk;
  }
  const int small = filter_table(g, ph || pw ? filter_taps(g, MNV_SMALL_TILE) : 1)
                        ? small_filter_ranges(g, N * (filter_positions(g) / 16), (size_t)-1) : 0;
  if (small > 1 && (size_t)small * g.CRS * K * sizeof(float) > bytes) bytes = (size_t)small * g.CRS * K * sizeof(float);
  if (mnv_wino_grad_images(N, C, K, H, W, ph, pw, R, S, sv, sh, (size_t)-1)) {
    const size_t w = mnv_wino_grad_workspace_bytes(N, C, K, H, W, ph, pw, R);
    if (w > bytes) bytes = w;
  }
  return bytes;
}

static int conv_bwd_filter_impl(const float* bottom, const float* top_diff, float* filter_diff,
                                int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh,
                                int R, int S, void* workspace, size_t workspace_bytes,
                                mnv_stream_t stream, int accumulate,
                                const float* sgd_w = nullptr, float sgd_scale = 0.f,
                                int* plan = nullptr) {
  ConvGeom g;
  if (!plan && (!bottom || !top_diff || !filter_diff)) return MNV_ERR_INVALID;
  int rc = make_geom(&g, N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (rc) return rc;
  int gm = g.CRS, gn = K, gk = N * g.HoWo;
  hipStream_t s = mnv_stream(stream);
  // 3 x 3 and 5 x 5 unit-stride layers with enough channels and tiles: minimal filtering of the
  // filter gradient, F(r x r, m x m), see winograd.hip
  if (const int images = mnv_wino_grad_images(N, C, K, H, W, ph, pw, R, S, sv, sh,
                                              workspace && (plan || mnv_aligned16(workspace)) ? workspace_bytes : 0))
    return mnv_wino_filter_grad(bottom, top_diff, filter_diff, N, C, K, H, W, ph, pw, R, images,
                                accumulate, sgd_w, sgd_scale, workspace, workspace_bytes, s, plan);
  int splits = bwd_filter_splits(gm, gn, gk, workspace ? workspace_bytes / sizeof(float) : 0);
  const int tile = bwd_filter_tile(gm, gn);
  // Fast addressing: rows in (tap, channel) order with per-tap offset tables in LDS.  The
  // tables of all taps a 128-row tile touches must fit beside the tiles.
  const int PP = filter_positions(g);
  // Sized exactly, conv2's tables (C = 96, 27 x 27 positions) take 5.9 KB instead of 8.8 KB, which is what
  // lets four workgroups share a CU's 160 KB of LDS.
  const int taps_per_block = filter_taps(g, 128);
  // On the small tiles, where they are the faster ones: sets `done`.
  auto small = [&](bool* done) -> int {
    const bool np = ph == 0 && pw == 0;
    const int taps = np ? 1 : filter_taps(g, MNV_SMALL_TILE), slabs = N * (PP / 16);
    const int z = filter_table(g, taps) ? small_filter_ranges(g, slabs, workspace ? workspace_bytes / sizeof(float) : 0) : 0;
    *done = z > 0;
    if (!z) return MNV_OK;
    if (plan) {
      plan[0] = MNV_SMALL_TILE;
      plan[1] = z;
      return MNV_OK;
    }
    if (np)
      return mnv_gemm_small_launch(ConvBwdFilterFast<true>{bottom, top_diff, filter_diff, g, gm, gn, gk, slabs, PP / 16, PP, 1,
                                                           mnv_fastdiv_make(C), accumulate, sgd_w, sgd_scale}, z, workspace, s);
    return mnv_gemm_small_launch(ConvBwdFilterFast<false>{bottom, top_diff, filter_diff, g, gm, gn, gk, slabs, PP / 16, PP, taps,
                                                          mnv_fastdiv_make(C), accumulate, sgd_w, sgd_scale}, z, workspace, s);
  };
  if (tile != 0 && ph == 0 && pw == 0 && (size_t)PP * 4 <= 24 * 1024) {
    ConvBwdFilterFast<true> p{bottom, top_diff, filter_diff, g, gm, gn, gk, N * (PP / 16),
                              PP / 16, PP, 1, mnv_fastdiv_make(C), accumulate, sgd_w, sgd_scale};
    return launch_filter_gradient<true>(tile, p, splits, workspace, workspace_bytes, s, plan, small);
  }
  if (tile != 0 && C % 128 == 0 && (size_t)PP * 4 <= 24 * 1024) {
    ConvBwdFilterFast<false, 1> p{bottom, top_diff, filter_diff, g, gm, gn, gk, N * (PP / 16),
                                  PP / 16, PP, 1, mnv_fastdiv_make(C), accumulate, sgd_w, sgd_scale};
    return launch_filter_gradient(tile, p, splits, workspace, workspace_bytes, s, plan, small);
  }
  if (tile != 0 && C % 16 == 0 && taps_per_block == 2 && (size_t)taps_per_block * PP * 4 <= 24 * 1024) {
    ConvBwdFilterFast<false, 3> p{bottom, top_diff, filter_diff, g, gm, gn, gk, N * (PP / 16),
                                  PP / 16, PP, taps_per_block, mnv_fastdiv_make(C), accumulate,
                                  sgd_w, sgd_scale};
    return launch_filter_gradient(tile, p, splits, workspace, workspace_bytes, s, plan, small);
  }
  if (tile != 0 && C % 16 == 0 && (size_t)taps_per_block * PP * 4 <= 24 * 1024) {
    ConvBwdFilterFast<false, 2> p{bottom, top_diff, filter_diff, g, gm, gn, gk, N * (PP / 16),
                                  PP / 16, PP, taps_per_block, mnv_fastdiv_make(C), accumulate,
                                  sgd_w, sgd_scale};
    return launch_filter_gradient(tile, p, splits, workspace, workspace_bytes, s, plan, small);
  }
  if (tile != 0 && (size_t)taps_per_block * PP * 4 <= 24 * 1024) {
    ConvBwdFilterFast<false> p{bottom, top_diff, filter_diff, g, gm, gn, gk, N * (PP / 16),
                               PP / 16, PP, taps_per_block, mnv_fastdiv_make(C), accumulate, sgd_w, sgd_scale};
    return launch_filter_gradient(tile, p, splits, workspace, workspace_bytes, s, plan, small);
  }
  ConvBwdFilter p{bottom, top_diff, filter_diff, g, gm, gn, gk, (gk + 15) / 16, 1, accumulate, sgd_w, sgd_scale};
  return launch_filter_gradient(tile, p, splits, workspace, workspace_bytes, s, plan, small);
}

int mnv_conv_bwd_filter(const float* bottom, const float* top_diff, float* filter_diff, int N,
                        int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R, int S,
                        void* workspace, size_t workspace_bytes, mnv_stream_t stream) {
  const int chunk = images_per_launch(N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (chunk <= 0 || chunk >= N)
    return conv_bwd_filter_impl(bottom, top_diff, filter_diff, N, C, K, H, W, ph, pw, sv, sh, R, S,
                                workspace, workspace_bytes, stream, 0);
  if (!bottom || !top_diff) return MNV_ERR_INVALID;
  const size_t per_bottom = (size_t)C * H * W;
  const size_t per_top = (size_t)K * ((H + 2 * ph - R) / sv + 1) * ((W + 2 * pw - S) / sh + 1);
  for (int n0 = 0; n0 < N; n0 += chunk) {
    const int nn = N - n0 < chunk ? N - n0 : chunk;
    int rc = conv_bwd_filter_impl(bottom + n0 * per_bottom, top_diff + n0 * per_top, filter_diff, nn,
                                  C, K, H, W, ph, pw, sv, sh, R, S, workspace, workspace_bytes,
                                  stream, n0 > 0);
    if (rc) return rc;
  }
  return MNV_OK;
}

static int direct_plan(bool forward, int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R, int S,
                       size_t workspace_bytes, DirectPlan* plan) {
  const int chunk = images_per_launch(N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (chunk <= 0) return MNV_ERR_INVALID;
  // the workspace is only compared with sizes here, never dereferenced
  void* some = workspace_bytes ? reinterpret_cast<void*>((uintptr_t)256) : nullptr;
  const int n = chunk < N ? chunk : N;
  return forward ? conv_fwd_impl(nullptr, nullptr, nullptr, nullptr, n, C, K, H, W, ph, pw, sv, sh, R, S, some, workspace_bytes,
                                 nullptr, 0, plan)
                 : conv_bwd_data_impl(nullptr, nullptr, nullptr, nullptr, n, C, K, H, W, ph, pw, sv, sh, R, S, some,
                                      workspace_bytes, nullptr, plan);
}

int mnv_conv_fwd_plan(int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R, int S, size_t workspace_bytes,
                      int* tile_rows, int* k_ranges, int* parts) {
  DirectPlan plan{};
  const int rc = direct_plan(true, N, C, K, H, W, ph, pw, sv, sh, R, S, workspace_bytes, &plan);
  if (rc) return rc;
  if (tile_rows) *tile_rows = plan.rows;
  if (k_ranges) *k_ranges = plan.ranges;
  if (parts) *parts = plan.parts;
  return MNV_OK;
}

int mnv_conv_bwd_data_plan(int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R, int S, size_t workspace_bytes,
                           int* tile_rows, int* k_ranges, int* parts, int* classes) {
  DirectPlan plan{};
  const int rc = direct_plan(false, N, C, K, H, W, ph, pw, sv, sh, R, S, workspace_bytes, &plan);
  if (rc) return rc;
  if (tile_rows) *tile_rows = plan.rows;
  if (k_ranges) *k_ranges = plan.ranges;
  if (parts) *parts = plan.parts;
  if (classes) *classes = plan.classes;
  return MNV_OK;
}

int mnv_conv_bwd_filter_plan(int N, int C, int K, int H, int W, int ph, int pw, int sv, int sh, int R,
                             int S, size_t workspace_bytes, int* tile_rows, int* k_ranges,
                             int* streamk_workgroups) {
  int plan[3] = {0, 0, 0};
  const int chunk = images_per_launch(N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (chunk <= 0) return MNV_ERR_INVALID;
  // the workspace is only compared with sizes here, never dereferenced
  void* some = workspace_bytes ? reinterpret_cast<void*>(&plan) : nullptr;
  int rc = conv_bwd_filter_impl(nullptr, nullptr, nullptr, chunk < N ? chunk : N, C, K, H, W, ph, pw, sv,
                                sh, R, S, some, workspace_bytes, nullptr, 0, nullptr, 0.f, plan);
  if (rc) return rc;
  if (tile_rows) *tile_rows = plan[0];
  if (k_ranges) *k_ranges = plan[1];
  if (streamk_workgroups) *streamk_workgroups = plan[2];
  return MNV_OK;
}

int mnv_conv_bwd_filter_sgd(const float* bottom, const float* top_diff, const float* filter,
                            float scale, float* filter_out, int N, int C, int K, int H, int W,
                            int ph, int pw, int sv, int sh, int R, int S, void* workspace,
                            size_t workspace_bytes, mnv_stream_t stream) {
  if (!filter || !filter_out) return MNV_ERR_INVALID;
  // a gradient summed over several launches cannot be folded into the store of one
  const int chunk = images_per_launch(N, C, K, H, W, ph, pw, sv, sh, R, S);
  if (chunk > 0 && chunk < N) return MNV_ERR_INVALID;
  return conv_bwd_filter_impl(bottom, top_diff, filter_out, N, C, K, H, W, ph, pw, sv, sh, R, S,
                              workspace, workspace_bytes, stream, 0, filter, scale);
}

}  // extern "C"
