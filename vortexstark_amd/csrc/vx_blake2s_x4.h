// Quad-parallel Blake2s (device only): the four lanes of a quad compute one
// compression together, lane q holding column q of the state (v[q], v[4+q],
// v[8+q], v[12+q]). The column step is one G per lane. For the diagonal step
// G's second operand stays where it is and the other three move: lane q takes
// v[q-1], v[8+q+1], v[12+q+2] (mod 4), which DPP quad permutes bring in and
// take back register to register, and runs diagonal q-1. (The second operand
// is G's last result: moving the earlier three keeps the permutes, and the
// two wait states a DPP read needs after a write, off the dependent chain.)
//
// A compression is 300 instructions per lane besides fetching message words:
//   b2_hash_x4      words in registers, selected by lane: 3 per word, ~430 in
//                   all. For dependent chains (tree tops, transcript): 0.73 us
//                   a level at four cycles per instruction of one wavefront.
//   b2_hash_x4_lds  the message in LDS, each lane reading its words at offsets
//                   fixed per lane (QuadOff): 1 per word, ~350 in all. For
//                   kernels bound by instruction issue; alone, the wait for
//                   the first words takes back what the selects cost (0.69 us
//                   a level, and the offsets' setup comes on top).
// Same function as b2_compress.
#pragma once
#include "vx_blake2s.h"

namespace vx {

// quad_perm controls: VX_DPP_ROTk gives lane q the value of lane (q + k) % 4
#define VX_DPP_ROT1 0x39  // [1,2,3,0]
#define VX_DPP_ROT2 0x4E  // [2,3,0,1]
#define VX_DPP_ROT3 0x93  // [3,0,1,2]

__device__ __forceinline__ uint32_t quad_rot(uint32_t x, int ctrl) {
  // ctrl must be a compile-time constant at every call site
  switch (ctrl) {
    case VX_DPP_ROT1: return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, VX_DPP_ROT1, 0xF, 0xF, true);
    case VX_DPP_ROT2: return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, VX_DPP_ROT2, 0xF, 0xF, true);
    default: return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, VX_DPP_ROT3, 0xF, 0xF, true);
  }
}

// x = word k of {A, B, C, D} by lane q (two bits -> three selects)
__device__ __forceinline__ uint32_t sel4(bool q0, bool q1, uint32_t A, uint32_t B, uint32_t C, uint32_t D) {
  const uint32_t lo = q0 ? B : A, hi = q0 ? D : C;
  return q1 ? hi : lo;
}

// Keeps a DPP move a move: folded into its user it would wait for that
// user's other operand too.
__device__ __forceinline__ uint32_t quad_moved(uint32_t x) {
  asm("" : "+v"(x));
  return x;
}

// Round of the quad; x, y are this lane's column step words, z, w its
// diagonal step's.
__device__ __forceinline__ void b2_round_x4(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d, uint32_t x, uint32_t y,
                                            uint32_t z, uint32_t w) {
  VX_B2_G(a, b, c, d, x, y);
  a = quad_rot(a, VX_DPP_ROT3);
  d = quad_moved(quad_rot(d, VX_DPP_ROT2));
  c = quad_moved(quad_rot(c, VX_DPP_ROT1));
  VX_B2_G(a, b, c, d, z, w);
  a = quad_rot(a, VX_DPP_ROT1);
  d = quad_moved(quad_rot(d, VX_DPP_ROT2));
  c = quad_moved(quad_rot(c, VX_DPP_ROT3));
}

// Index in the message of word k of lane q's schedule: words 4r, 4r + 1 are
// round r's column step's, 4r + 2, 4r + 3 its diagonal step's.
__host__ __device__ constexpr uint32_t quad_word(uint32_t q, uint32_t k) {
  return B2_SIGMA[k / 4][k % 4 < 2 ? 2 * q + k % 4 : 8 + 2 * ((q + 3) % 4) + k % 4 - 2];
}

// The ten rounds on a message in registers (the quad passes the same words).
struct QuadRegs {
  const uint32_t (&m)[16];
  const bool q0, q1;
  __device__ __forceinline__ uint32_t word(int k) const {
    return sel4(q0, q1, m[quad_word(0, k)], m[quad_word(1, k)], m[quad_word(2, k)], m[quad_word(3, k)]);
  }
  __device__ __forceinline__ void rounds(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) const {
#pragma unroll
    for (int r = 0; r < 10; r++)
      b2_round_x4(a, b, c, d, word(4 * r), word(4 * r + 1), word(4 * r + 2), word(4 * r + 3));
  }
};

// Byte offsets of a lane's schedule words in an LDS message, the quad's
// message at byte offset `at`. Node messages lie QUAD_STRIDE words apart: 16
// words and 4 of padding, so that the lanes of a wavefront reading the same
// word of their nodes spread over the banks.
static constexpr uint32_t QUAD_STRIDE = 20;
struct QuadOff {
  uint32_t off[40];
};
struct QuadOffTable {
  uint4 b[4][3];  // lane q: byte offsets (4 * word), one byte each, 40 of 48 used
};
constexpr QuadOffTable make_quad_off_table() {
  QuadOffTable t{};
  for (uint32_t q = 0; q < 4; q++) {
    uint32_t w[12] = {};
    for (uint32_t k = 0; k < 40; k++) w[k / 4] |= (4 * quad_word(q, k)) << (8 * (k % 4));
    for (uint32_t v = 0; v < 3; v++) {
      t.b[q][v].x = w[4 * v];
      t.b[q][v].y = w[4 * v + 1];
      t.b[q][v].z = w[4 * v + 2];
      t.b[q][v].w = w[4 * v + 3];
    }
  }
  return t;
}
__constant__ const QuadOffTable QUAD_OFF_TABLE = make_quad_off_table();

// The table row of a lane, fetched ahead of its use, and the offsets from it.
struct QuadRow {
  uint4 x, y;
  uint2 z;
};
__device__ __forceinline__ QuadRow quad_row(uint32_t q) {
  const uint4 z = QUAD_OFF_TABLE.b[q][2];
  return {QUAD_OFF_TABLE.b[q][0], QUAD_OFF_TABLE.b[q][1], make_uint2(z.x, z.y)};
}
__device__ __forceinline__ QuadOff quad_off(const QuadRow& t, uint32_t at) {
  const uint32_t w[10] = {t.x.x, t.x.y, t.x.z, t.x.w, t.y.x, t.y.y, t.y.z, t.y.w, t.z.x, t.z.y};
  QuadOff o;
#pragma unroll
  for (int k = 0; k < 40; k++) o.off[k] = at + ((w[k / 4] >> (8 * (k % 4))) & 0xFFu);
  return o;
}
// The ten rounds on a message in LDS. A round's words are read two rounds
// ahead (about 60 instructions, 240 cycles); left to itself the compiler reads
// each word five instructions before its use and waits for it 40 times.
struct QuadLds {
  const uint32_t* msg;
  const QuadOff& o;
  __device__ __forceinline__ void rounds(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) const {
    constexpr int AHEAD = 2;
    uint32_t w[40];
    auto read = [&](int r) {
#pragma unroll
      for (int k = 4 * r; k < 4 * r + 4; k++)
        w[k] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(msg) + o.off[k]);
    };
#pragma unroll
    for (int r = 0; r < AHEAD; r++) read(r);
#pragma unroll
    for (int r = 0; r < 10; r++) {
      if (r + AHEAD < 10) read(r + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      b2_round_x4(a, b, c, d, w[4 * r], w[4 * r + 1], w[4 * r + 2], w[4 * r + 3]);
    }
  }
};

// The ten rounds on a message a lane holds in its own schedule order.
struct QuadSched {
  const uint4 (&w)[10];
  __device__ __forceinline__ void rounds(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) const {
#pragma unroll
    for (int r = 0; r < 10; r++) b2_round_x4(a, b, c, d, w[r].x, w[r].y, w[r].z, w[r].w);
  }
};

// Single-block Blake2s of `t` message bytes (the final block; bytes past t
// are zero in the message) by the four lanes of a quad, q = lane & 3. Returns
// output words q and 4 + q in lo / hi.
template <typename W>
__device__ __forceinline__ void b2_final_x4(const W& w, uint32_t t, uint32_t q, uint32_t& lo, uint32_t& hi) {
  const bool q0 = q & 1, q1 = q & 2;
  const uint32_t iv_lo = sel4(q0, q1, VX_B2_IV0, VX_B2_IV1, VX_B2_IV2, VX_B2_IV3);
  const uint32_t iv_hi = sel4(q0, q1, VX_B2_IV4, VX_B2_IV5, VX_B2_IV6, VX_B2_IV7);
  const uint32_t h_lo = q == 0 ? VX_B2_H0 : iv_lo, h_hi = iv_hi;
  uint32_t a = h_lo, b = h_hi, c = iv_lo;
  uint32_t d = iv_hi ^ (q == 0 ? t : 0u) ^ (q == 2 ? 0xFFFFFFFFu : 0u);  // v12 ^= t, v14 ^= final
  w.rounds(a, b, c, d);
  lo = h_lo ^ a ^ c;
  hi = h_hi ^ b ^ d;
}
__device__ __forceinline__ void b2_hash_x4(const uint32_t (&m)[16], uint32_t t, uint32_t q, uint32_t& lo, uint32_t& hi) {
  b2_final_x4(QuadRegs{m, (q & 1) != 0, (q & 2) != 0}, t, q, lo, hi);
}
__device__ __forceinline__ void b2_hash_x4_lds(const uint32_t* msg, const QuadOff& o, uint32_t t, uint32_t q,
                                               uint32_t& lo, uint32_t& hi) {
  b2_final_x4(QuadLds{msg, o}, t, q, lo, hi);
}

// One compression of a chained hash by the four lanes of a quad: lane q
// holds chaining words q and 4 + q in h_lo / h_hi and updates them; t is the
// byte count up to and including this block, last marks the final block.
// All four lanes pass the same 16 message words, or each its own schedule of
// them. Same function as b2_compress.
template <typename W>
__device__ __forceinline__ void b2_compress_x4_of(uint32_t& h_lo, uint32_t& h_hi, const W& words, uint32_t t, bool last,
                                                  uint32_t q) {
  const bool q0 = q & 1, q1 = q & 2;
  uint32_t a = h_lo, b = h_hi;
  uint32_t c = sel4(q0, q1, VX_B2_IV0, VX_B2_IV1, VX_B2_IV2, VX_B2_IV3);
  uint32_t d = sel4(q0, q1, VX_B2_IV4, VX_B2_IV5, VX_B2_IV6, VX_B2_IV7) ^ (q == 0 ? t : 0u) ^
               (q == 2 && last ? 0xFFFFFFFFu : 0u);  // v12 ^= t, v14 ^= final
  words.rounds(a, b, c, d);
  h_lo ^= a ^ c;
  h_hi ^= b ^ d;
}
__device__ __forceinline__ void b2_compress_x4(uint32_t& h_lo, uint32_t& h_hi, const uint32_t (&m)[16], uint32_t t,
                                               bool last, uint32_t q) {
  b2_compress_x4_of(h_lo, h_hi, QuadRegs{m, (q & 1) != 0, (q & 2) != 0}, t, last, q);
}
__device__ __forceinline__ void b2_compress_x4(uint32_t& h_lo, uint32_t& h_hi, const uint4 (&w)[10], uint32_t t,
                                               bool last, uint32_t q) {
  b2_compress_x4_of(h_lo, h_hi, QuadSched{w}, t, last, q);
}

// LDS writes of a lane before, LDS reads of the wavefront's other lanes
// after: the LDS unit keeps one wavefront's accesses in order, so only the
// compiler has to.
__device__ __forceinline__ void wave_lds_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// Merkle node hash (t = 64).
__device__ __forceinline__ void b2_node_x4(const uint32_t (&m)[16], uint32_t q, uint32_t& lo, uint32_t& hi) {
  b2_hash_x4(m, 64u, q, lo, hi);
}

// The 8 output words of a quad hash in every lane of the quad: word k
// (k < 4) is lane k's lo, word 4 + k its hi. The quad must be lanes 0..3 of
// the wavefront (readlane reads fixed lanes).
__device__ __forceinline__ void quad0_gather(uint32_t lo, uint32_t hi, uint32_t out[8]) {
#pragma unroll
  for (int k = 0; k < 4; k++) {
    out[k] = (uint32_t)__builtin_amdgcn_readlane((int)lo, k);
    out[4 + k] = (uint32_t)__builtin_amdgcn_readlane((int)hi, k);
  }
}

}  // namespace vx
