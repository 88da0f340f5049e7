// The largest span of a launch (wino_most_of_spans) against a walk over all of its workgroups, on random
// planes, batches and tiles; every workgroup's tiles lie inside its span; and the number of workgroups looked
// at does not grow with the batch.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "winograd_spans.h"

namespace {

int failures = 0;
void check(bool ok, const char* what) {
  if (!ok && failures++ < 5) std::printf("FAILED: %s\n", what);
}

template <class Span>
int walk(int P, int TH, int TW, const Span& span) {
  const int T = TH * TW;
  int most = 0;
  for (int p0 = 0; p0 < P; p0 += 256) {
    const int last = p0 + 255 < P ? p0 + 255 : P - 1;
    const int a = p0 / T, b = last / T;
    const WinoSpan s = span((p0 - a * T) / TW, (last - b * T) / TW, b - a + 1);
    if (s.hi - s.lo > most) most = s.hi - s.lo;
  }
  return most;
}

template <class Span>
void compare(int P, int TH, int TW, int limit, const Span& span) {
  const int all = walk(P, TH, TW, span), got = wino_most_of_spans(P, TH, TW, limit, span);
  check(all > limit ? got == limit + 1 : got == all, "largest span");
}

}  // namespace

int main() {
  std::mt19937 rng(7);
  auto pick = [&](int n) { return (int)(rng() % (unsigned)n); };
  const int tiles[4][2] = {{4, 3}, {6, 3}, {7, 3}, {8, 5}};
  for (int it = 0; it < 60000; ++it) {
    const int* t = tiles[pick(4)];
    const int al = t[0], r = t[1], m = al - r + 1;
    const int H = 1 + pick(pick(4) ? 40 : 300), W = 1 + pick(pick(4) ? 40 : 300), pad = pick(r);
    const int Hd = H + 2 * pad - (r - 1), Wd = W + 2 * pick(r) - (r - 1);
    if (Hd <= 0 || Wd <= 0) continue;
    const int TH = (Hd + m - 1) / m, TW = (Wd + m - 1) / m, T = TH * TW, N = 1 + pick(300);
    if ((long long)N * T > 200000) continue;
    const int P = N * T, chunks = (H * W + 3) / 4;
    auto in = [&](int a, int b, int i) { return wino_span(a, b, i, m, pad, al, H, W, chunks); };
    auto grad = [&](int a, int b, int i) { return wino_span(a, b, i, m, 0, m, Hd, Wd, (Hd * Wd + 3) / 4); };
    auto out = [&](int a, int b, int i) { return wino_rows_span(a, b, i, m, Hd, Wd); };
    compare(P, TH, TW, 3072, in);
    compare(P, TH, TW, 3072, grad);
    compare(P, TH, TW, 12288, out);
    // one workgroup's tiles: every row of the plane that a tile reads is inside the span
    const int p0 = pick((P + 255) / 256) * 256, last = p0 + 255 < P ? p0 + 255 : P - 1, img0 = p0 / T;
    const WinoSpan s = in((p0 - img0 * T) / TW, (last - last / T * T) / TW, last / T - img0 + 1);
    for (int p = p0; p <= last; ++p)
      for (int a = 0; a < al; ++a) {
        const int y = m * (p % T / TW) - pad + a, base = (p / T - img0) * chunks;
        if (y >= 0 && y < H)
          check(base + y * W / 4 >= s.lo && base + (y * W + W - 1) / 4 < s.hi, "a tile's row outside its workgroup's span");
      }
  }
  int looked = 0;
  auto counted = [&](int a, int b, int i) {
    ++looked;
    return wino_rows_span(a, b, i, 4, 56, 56);
  };
  wino_most_of_spans(196 << 20, 14, 14, 12288, counted);
  check(looked <= 49, "workgroups looked at");
  if (failures) return 1;
  std::printf("OK\n");
  return 0;
}
