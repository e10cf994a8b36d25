// Stream-K split of W tiles over G work-groups (decode_main, decode_reduce),
// also compiled for the host by the test of its arithmetic.
#pragma once

#include <math.h>
#include <stdint.h>

namespace sia {

// The most work-groups of a split: sk_lo's products stay below 2^24.
constexpr int kMaxSplitGroups = 4095;

// Group g takes [lo(g), lo(g+1)) with lo(g) = floor(g W / G).  With W = Q G + R
// this is g Q + floor(g R / G), and g R < G^2 <= kMaxSplitGroups^2 stays below
// 2^24, where one fp32 product and a correction divide exactly.  (The 64-bit
// divisions this replaces took ~0.4 us of every group's start at one sequence
// of 1000 tokens.)
struct SkSplit {
  int W, G, Q, R;
  float rG, rW;        // 1 / G, 1 / W, each within an ulp
};
__host__ __device__ __forceinline__ SkSplit sk_split(int W, int G, float rG, float rW) {
  SkSplit s;
  s.W = W;
  s.G = G;
  s.Q = (int)((uint32_t)W / (uint32_t)G);
  s.R = W - s.Q * G;
  s.rG = rG;
  s.rW = rW;
  return s;
}
__host__ __device__ __forceinline__ int sk_lo(const SkSplit& s, int g) {
  const int n = g * s.R;
  int q = (int)((float)n * s.rG);
  const int r = n - q * s.G;
  q += r >= s.G ? 1 : r < 0 ? -1 : 0;
  return g * s.Q + q;
}
// The group holding position x (0 <= x < W), the last one with lo(g) <= x:
// ceil((x + 1) G / W) - 1 by an fp32 estimate, within one of it (the error is
// below G 2^-21), set right by the bounds.
__host__ __device__ __forceinline__ int sk_group(const SkSplit& s, int x) {
  int g = (int)ceilf((float)(x + 1) * ((float)s.G * s.rW)) - 1;
  g = g < 0 ? 0 : g > s.G - 1 ? s.G - 1 : g;
  if (g > 0 && sk_lo(s, g) > x) --g;
  if (g + 1 < s.G && sk_lo(s, g + 1) <= x) ++g;
  return g;
}

}  // namespace sia
