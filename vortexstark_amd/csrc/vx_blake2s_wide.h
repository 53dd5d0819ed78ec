// Blake2s compression for kernels with several wavefronts per SIMD (device
// only): the same function as b2_compress, ordered so that wavefronts issue
// together.
//
// How that works is described in vx_issue.h.
//
// So the four G of a half round advance together, their slow operations in
// groups of four or eight under raised priority. 480 of a compression's 960
// instructions are slow. Measured, 8,192 workgroups of 256: 38-39 -> 63
// giga-compressions/s (2 wavefronts per SIMD: 33 -> 40; one: 31 -> 24, so the
// latency-bound kernels keep b2_compress). Fibonacci log_n = 24: trace tree
// 3,495 -> 2,150 us, circle fold 1,860 -> 1,360 us, proof 11.95 -> 8.3 ms.
#pragma once
#include "vx_blake2s.h"
#include "vx_issue.h"

namespace vx {

namespace b2w {
using namespace issue;

// v[i] += v[b_i] + message word, the four G of half round `hr` (even: columns,
// odd: diagonals), word `k` (0 or 1) of each G. Words from NZ up are zero:
// those sums are plain adds, after the slow group.
template <uint32_t NZ>
__device__ __forceinline__ void add_words(uint32_t (&v)[16], const uint32_t (&m)[16], uint32_t hr, uint32_t k,
                                          bool slow) {
#pragma unroll
  for (uint32_t i = 0; i < 4; i++) {
    const uint32_t w = B2_SIGMA[hr / 2][8 * (hr % 2) + 2 * i + k], b = 4 + (i + hr % 2) % 4;
    if (slow && w < NZ) add3(v[i], v[b], m[w]);
    if (!slow && w >= NZ) add(v[i], v[b]);
  }
}
}  // namespace b2w

// The half rounds from FIRST on (0: all) of the working state v; words of m
// from NZ up are taken as zero.
template <uint32_t NZ, uint32_t FIRST>
__device__ __forceinline__ void b2_rounds_wide(uint32_t (&v)[16], const uint32_t (&m)[16]) {
  using namespace b2w;
  slow_begin();
  add_words<NZ>(v, m, FIRST, 0, true);
  slow_end();
  add_words<NZ>(v, m, FIRST, 0, false);
#pragma unroll
  for (uint32_t hr = FIRST; hr < 20; hr++) {
    const uint32_t g = hr % 2;  // G i works on v[i], v[4 + (i + g) % 4], v[8 + (i + 2 g) % 4], v[12 + (i + 3 g) % 4]
#pragma unroll
    for (uint32_t k = 0; k < 2; k++) {
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) eor(v[12 + (i + 3 * g) % 4], v[i]);
      slow_begin();
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) {
        if (k == 0) rot<16>(v[12 + (i + 3 * g) % 4]);
        else rot<8>(v[12 + (i + 3 * g) % 4]);
      }
      slow_end();
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) add(v[8 + (i + 2 * g) % 4], v[12 + (i + 3 * g) % 4]);
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) eor(v[4 + (i + g) % 4], v[8 + (i + 2 * g) % 4]);
      // the rotation of b and the sums that it feeds, of this half round or the next
      const bool more = k == 0 || hr < 19;
      const uint32_t nhr = k == 0 ? hr : hr + 1, nk = k == 0 ? 1 : 0;
      slow_begin();
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) {
        if (k == 0) rot<12>(v[4 + (i + g) % 4]);
        else rot<7>(v[4 + (i + g) % 4]);
      }
      if (more) add_words<NZ>(v, m, nhr, nk, true);
      slow_end();
      if (more) add_words<NZ>(v, m, nhr, nk, false);
    }
  }
}

__device__ __forceinline__ void b2_state(uint32_t (&v)[16], const uint32_t (&h)[8], uint32_t t, bool last) {
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = h[i];
  v[8] = VX_B2_IV0;
  v[9] = VX_B2_IV1;
  v[10] = VX_B2_IV2;
  v[11] = VX_B2_IV3;
  v[12] = VX_B2_IV4 ^ t;
  v[13] = VX_B2_IV5;
  v[14] = last ? ~VX_B2_IV6 : VX_B2_IV6;
  v[15] = VX_B2_IV7;
}

// h <- compress(h, m, t, last); words of m from NZ up are taken as zero.
template <uint32_t NZ = 16>
__device__ __forceinline__ void b2_compress_wide(uint32_t (&h)[8], const uint32_t (&m)[16], uint32_t t, bool last) {
  uint32_t v[16];
  b2_state(v, h, t, last);
  b2_rounds_wide<NZ, 0>(v, m);
#pragma unroll
  for (int i = 0; i < 8; i++) h[i] ^= v[i] ^ v[8 + i];
}

// b2_hash_words, b2_hash_node, b2_leaf1 and b2_leaf4 on it.
__device__ __forceinline__ void b2_hash_words_wide(const uint32_t* w, uint32_t nwords, uint32_t (&out)[8]) {
  uint32_t m[16];
#pragma unroll
  for (int i = 0; i < 16; i++) m[i] = (uint32_t)i < nwords ? w[i] : 0u;
  b2_init(out);
  b2_compress_wide(out, m, 4u * nwords, true);
}
__device__ __forceinline__ void b2_hash_node_wide(const uint32_t* l, const uint32_t* r, uint32_t (&out)[8]) {
  uint32_t m[16];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    m[i] = l[i];
    m[8 + i] = r[i];
  }
  b2_init(out);
  b2_compress_wide(out, m, 64u, true);
}
__device__ __forceinline__ void b2_leaf1_wide(uint32_t x, uint32_t (&out)[8]) {
  const uint32_t m[16] = {x};
  b2_init(out);
  b2_compress_wide<1>(out, m, 4u, true);
}
__device__ __forceinline__ void b2_leaf4_wide(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t (&out)[8]) {
  const uint32_t m[16] = {a, b, c, d};
  b2_init(out);
  b2_compress_wide<4>(out, m, 16u, true);
}

}  // namespace vx
