// Packing of the shape tree's nodes (layouts in isect.h).
#pragma once
#include <cmath>
#include <cstring>

#include "isect.h"

namespace bgpu {

inline uint32_t word_of(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return u;
}

// The half at or below x (down), or at or above it; an undefined plane bounds
// nothing.
inline uint32_t half_outward(float x, bool down) {
  if (x != x) return down ? 0xfc00u : 0x7c00u;
  const uint32_t u = word_of(x), sign = (u >> 16) & 0x8000u, m = u & 0x7fffffffu;
  const bool away = (sign != 0u) == down;  // the magnitude rounds up
  uint32_t h, rest;
  if (m >= 0x47800000u) {  // 65536 and more, and infinity
    h = m == 0x7f800000u ? 0x7c00u : 0x7bffu;
    rest = m == 0x7f800000u ? 0u : 1u;
  } else if (m >= 0x38800000u) {  // normal halves, from 2^-14
    h = (m - 0x38000000u) >> 13;
    rest = m & 0x1fffu;
  } else {  // subnormal halves: multiples of 2^-24
    const uint32_t e = m >> 23, f = (m & 0x7fffffu) | (e ? 0x800000u : 0u), shift = 126u - e;
    h = shift < 25u ? f >> shift : 0u;
    rest = shift < 25u ? f & ((1u << shift) - 1u) : f;
  }
  return sign | (h + (away && rest ? 1u : 0u));
}

// The nearest float at or below (down), or at or above d.
inline float float_outward(double d, bool down) {
  const float f = (float)d;
  if (down ? (double)f > d : (double)f < d) return nextafterf(f, down ? -INFINITY : INFINITY);
  return f;
}

inline uint32_t bf16_up(float x) {  // x >= 0, or NaN (taken as +inf)
  return x < INFINITY ? (word_of(x) + 0xffffu) >> 16 : 0x7f80u;
}

// Node `o` of 8 * W floats to node_words(W) words.  The differences to
// the centre are taken in binary64, where they are exact or off by far less
// than a half's step.
template <int W>
inline void pack_node(const float* o, float scale, uint32_t* v) {
  float r2 = 0.0f;
  for (int k = 0; k < 3; ++k) {
    const float *lo = o + 2 * k * W, *hi = lo + W;
    float a = lo[0], b = hi[0];
    for (int c = 1; c < W; ++c) {
      a = fminf(a, lo[c]);
      b = fmaxf(b, hi[c]);
    }
    float org = 0.5f * a + 0.5f * b;
    if (!(fabsf(org) < INFINITY)) org = 0.0f;
    const float half = fmaxf(org - a, b - org) * 1.0001f;
    r2 += half * half;
    for (int c = 0; c < W; c += 2) {
      uint32_t wl = 0u, wh = 0u;
      for (int q = 0; q < 2; ++q) {
        wl |= half_outward(float_outward(((double)lo[c + q] - org) * scale, true), true) << (16 * q);
        wh |= half_outward(float_outward(((double)hi[c + q] - org) * scale, false), false) << (16 * q);
      }
      v[4 + k * W + c / 2] = wl;
      v[4 + k * W + W / 2 + c / 2] = wh;
    }
    v[k] = word_of(org);
  }
  float h = o[7 * W];
  for (int c = 1; c < W; ++c) h = fmaxf(h, o[7 * W + c]);
  v[3] = bf16_up(sqrtf(r2) * 1.0001f) << 16 | bf16_up(h);
  for (int c = 0; c < W; ++c) v[4 + 3 * W + c] = word_of(o[6 * W + c]);
}

}  // namespace bgpu
