// What of the image planes the 256 tiles of a workgroup need in LDS (winograd.hip's transform kernels),
// computed alike by the kernels and by the host that sizes their LDS.
#pragma once
#ifdef __HIPCC__
#define MNV_HOST_DEVICE __host__ __device__
#else
#define MNV_HOST_DEVICE
#endif

// What of the planes the 256 tiles from p0 on read, in 16-byte chunks: chunk c of plane i of
// the tiles' images (the first one's plane is 0) is number i chunks + c, chunks = ceil(HW / 4),
// and the tiles need the numbers [lo, hi) -- of the first and the last image only the rows that
// hold their tiles.  A tile row th needs the plane's rows from m th - pad on, `reach` of them.
struct WinoSpan {
  int lo, hi;
};
MNV_HOST_DEVICE inline WinoSpan wino_span(int th0, int th1, int images, int m, int pad, int reach, int H, int W,
                                          int chunks) {
  const int y0 = m * th0 - pad > 0 ? m * th0 - pad : 0;
  const int y1 = m * th1 - pad + reach < H ? m * th1 - pad + reach : H;
  return WinoSpan{y0 * W / 4, (images - 1) * chunks + (y1 * W + 3) / 4};
}

// The same of the output planes, laid end to end, in floats: the rows that the tiles cover.
MNV_HOST_DEVICE inline WinoSpan wino_rows_span(int th0, int th1, int images, int m, int H, int W) {
  return WinoSpan{m * th0 * W, (images - 1) * H * W + (m * (th1 + 1) < H ? m * (th1 + 1) : H) * W};
}

// The largest span of a launch's workgroups, or `limit` + 1 as soon as one is past the limit:
// span(first tile row, last tile row, images).  Where a workgroup's tiles begin in a plane repeats
// after T / gcd(T, 256) workgroups, and one that the last tile cuts spans no more than a whole one.
template <class Span>
int wino_most_of_spans(int P, int TH, int TW, int limit, const Span& span) {
  const int T = TH * TW, groups = (P + 255) / 256;
  int period = T;
  for (int f = 256; f > 1 && period % 2 == 0; f /= 2) period /= 2;
  int most = 0;
  for (int i = 0; i < (groups < period ? groups : period); ++i) {
    const int p0 = 256 * i, last = p0 + 255 < P ? p0 + 255 : P - 1;
    const int img0 = p0 / T, img1 = last / T;
    const WinoSpan s = span((p0 - img0 * T) / TW, (last - img1 * T) / TW, img1 - img0 + 1);
    if (s.hi - s.lo > limit) return limit + 1;
    if (s.hi - s.lo > most) most = s.hi - s.lo;
  }
  return most;
}
