// Device-resident Fiat-Shamir transcript and deterministic PoW grind.
//
// The transcript (src/channel.rs:15-185) runs on the GPU so a whole proof is
// one stream of kernels with no host round trip: each commitment root is
// mixed by a single lane, and the next fold reads its alpha from device
// memory. Query draws are independent squeezes (n_draws = 0..nq-1 after
// mix_felts), so one lane per query computes them in parallel.
#include "vx_blake2s_wide.h"
#include "vx_blake2s_x4.h"
#include "vx_internal.h"

namespace vx {

__global__ void k_channel_step(Channel* ch, int init, const uint32_t* digest, uint32_t* alpha_out,
                               uint32_t* alpha_sq_out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  Channel c;
  if (init) ch_init(c);
  else c = *ch;
  if (digest) {
    uint32_t d[8];
    for (int k = 0; k < 8; k++) d[k] = digest[k];
    ch_mix_digest(c, d);
  }
  if (alpha_out) {
    qm31 a = ch_draw_felt(c);
    for (int k = 0; k < 4; k++) alpha_out[k] = a.v[k];
    if (alpha_sq_out) {
      qm31 a2 = qm_mul(a, a);
      for (int k = 0; k < 4; k++) alpha_sq_out[k] = a2.v[k];
    }
  }
  *ch = c;
}

void channel_step(Channel* ch, bool init, const uint32_t* digest, uint32_t* alpha_out, uint32_t* alpha_sq_out,
                  hipStream_t s) {
  hipLaunchKernelGGL(k_channel_step, dim3(1), dim3(64), 0, s, ch, init ? 1 : 0, digest, alpha_out, alpha_sq_out);
  VX_HIP(hipGetLastError());
}

// mix_felts(last layer) (src/prover.rs:554); writes n_last + the 8 values
// into the proof. With PoW: the prefix digest of the new state, and the search's
// nonce set to "none". Without: the queries too, when one workgroup's lanes
// cover them (MIX_QUERIES_MAX), so that the step is one launch.
//
// A dependent chain of three or four compressions: by the quad of lanes 0..3 on
// words in LDS: 6.0 us with the queries, where one lane took 7.7 us and the
// queries a launch of 4.4 us more.
static constexpr uint32_t MIX_THREADS = 256, MIX_QUERIES_MAX = MIX_THREADS;

__device__ __forceinline__ void draw_query(const QueryArgs& q, Channel c, uint32_t i) {
  c.n_draws = i;
  const uint32_t v = (uint32_t)ch_draw_number(c, q.domain);
  q.queries[i] = v;
  q.proof[q.query_word + 1 + i] = v;
}

__global__ __launch_bounds__(MIX_THREADS) void k_mix_last(QueryArgs q, uint32_t* prefix_out, uint64_t* nonce_out) {
  __shared__ uint32_t msg[48];  // state || 8 QM31 values, zero-padded to whole blocks
  __shared__ uint32_t state[8];
  const uint32_t tid = threadIdx.x;
  if (tid < 8) {
    msg[tid] = q.ch->state[tid];
  } else if (tid < 40) {
    const uint32_t i = tid - 8, v = q.last[i & 3][i >> 2];
    msg[tid] = v;
    q.proof[q.last_word + 1 + i] = v;
  } else if (tid < 48) {
    msg[tid] = 0;
  } else if (tid == 48) {
    q.proof[q.last_word] = 8;
    if (!q.pow_bits) q.proof[q.query_word] = q.nq;
  }
  __syncthreads();
  if (tid < 64) {
    const uint32_t l = tid & 3;
    const bool q0 = l & 1, q1 = l & 2;
    uint32_t lo = sel4(q0, q1, VX_B2_H0, VX_B2_IV1, VX_B2_IV2, VX_B2_IV3);
    uint32_t hi = sel4(q0, q1, VX_B2_IV4, VX_B2_IV5, VX_B2_IV6, VX_B2_IV7);
    uint32_t m[16];
    for (uint32_t blk = 0; blk < 3; blk++) {
#pragma unroll
      for (int k = 0; k < 16; k++) m[k] = msg[16 * blk + k];
      b2_compress_x4(lo, hi, m, blk < 2 ? 64 * (blk + 1) : 160u, blk == 2, l);
    }
    if (tid < 4) {
      state[l] = lo;
      state[4 + l] = hi;
      q.ch->state[l] = lo;
      q.ch->state[4 + l] = hi;
    }
    if (tid == 0) q.ch->n_draws = 0;
    if (q.pow_bits && prefix_out) {  // ch_pow_prefix
      wave_lds_order();
#pragma unroll
      for (int k = 0; k < 16; k++) m[k] = k == 0 ? 0x12345678u : k == 12 ? q.pow_bits : k >= 4 && k < 12 ? state[k - 4] : 0u;
      b2_hash_x4(m, 52u, l, lo, hi);
      if (tid < 4) {
        prefix_out[l] = lo;
        prefix_out[4 + l] = hi;
      }
      if (tid == 0) *nonce_out = ~0ull;
    }
  }
  if (q.pow_bits || q.nq > MIX_QUERIES_MAX) return;
  __syncthreads();
  if (tid < q.nq) {
    Channel c;
#pragma unroll
    for (int k = 0; k < 8; k++) c.state[k] = state[k];
    draw_query(q, c, tid);
  }
}

// Query i is draw_number(domain) at n_draws = i (src/prover.rs:555-557),
// after mix_u64(nonce) when PoW is on.
__global__ void k_draw_queries(QueryArgs q) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  Channel c = *q.ch;
  if (q.pow_bits) {
    uint64_t nonce = *q.nonce;
    ch_mix_u64(c, nonce);
    if (i == 0) {
      q.proof[q.nonce_word] = (uint32_t)nonce;
      q.proof[q.nonce_word + 1] = (uint32_t)(nonce >> 32);
    }
  }
  if (i == 0) q.proof[q.query_word] = q.nq;
  if (i < q.nq) draw_query(q, c, i);
}

void channel_queries(const QueryArgs& q, uint32_t* prefix, uint64_t* nonce, hipStream_t s) {
  require(q.nq >= 1 && q.nq <= 65536, "queries: 1..65536 queries");
  hipLaunchKernelGGL(k_mix_last, dim3(1), dim3(MIX_THREADS), 0, s, q, prefix, nonce);
  VX_HIP(hipGetLastError());
  if (q.pow_bits) grind_pow(prefix, q.pow_bits, nonce, s, true);
  if (!q.pow_bits && q.nq <= MIX_QUERIES_MAX) return;
  hipLaunchKernelGGL(k_draw_queries, dim3((q.nq + 255) / 256), dim3(256), 0, s, q);
  VX_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ PoW
// Nonces are scanned in increasing order by a grid-stride loop; every lane
// keeps going while its next nonce is below the best found so far, so every
// nonce smaller than the final answer has been tested: the result is the
// smallest valid nonce, independent of scheduling. Each wave reduces its
// hits with a wavefront min before one atomicMin.
static constexpr uint64_t GRIND_LIMIT = 1ull << 44;  // exit bound every lane reaches

__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    uint64_t o = __shfl_xor(v, off, 64);
    v = o < v ? o : v;
  }
  return v;
}

// The stwo plugin's nonce family (crates/cuda-backend/src/grind_ops.rs:
// 71-128): index i stands for nonce ((i >> 20) << 32) | (i & (2^20 - 1)), a
// map that keeps the order, so the smallest index is the smallest nonce.
__device__ __forceinline__ uint64_t stwo_nonce(uint64_t i) { return ((i >> 20) << 32) | (i & 0xFFFFFull); }

// WIDE (grids of at least two wavefronts per SIMD): b2_compress_wide's half
// rounds. The first one mixes the prefix only, so it is done once per lane
// and not per nonce. PoW 20 (about 2^20 nonces, 1,024 workgroups): 20.0 ->
// 17.9 us.
template <bool STWO, bool M31_OUT, bool WIDE>
__global__ __launch_bounds__(256) void k_grind(const uint32_t* prefix_dev, uint32_t bits,
                                              unsigned long long* best, uint64_t start, uint64_t count) {
  uint32_t prefix[8];
  for (int k = 0; k < 8; k++) prefix[k] = prefix_dev[k];
  uint32_t h0[8], v0[16];
  b2_init(h0);
  b2_state(v0, h0, 40u, true);
#pragma unroll
  for (int i = 0; i < 4; i++) VX_B2_G(v0[i], v0[4 + i], v0[8 + i], v0[12 + i], prefix[2 * i], prefix[2 * i + 1]);
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t end = start + count;
  for (uint64_t base = start + (uint64_t)blockIdx.x * blockDim.x; base < end; base += stride) {
    // Wave-uniform exit: lane 0's view of the best hit decides for the wave,
    // so the shuffles below always run with all 64 lanes active.
    const uint64_t seen = __hip_atomic_load(best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t cur_best = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(seen >> 32)) << 32) |
                              (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)seen);
    if (base > cur_best) break;
    const uint64_t n = base + threadIdx.x;
    const uint64_t nonce = STWO ? stwo_nonce(n) : n;
    uint32_t tz;
    if constexpr (WIDE) {
      const uint32_t m[16] = {prefix[0], prefix[1], prefix[2], prefix[3],     prefix[4],
                              prefix[5], prefix[6], prefix[7], (uint32_t)nonce, (uint32_t)(nonce >> 32)};
      uint32_t v[16], h[4];
#pragma unroll
      for (int i = 0; i < 16; i++) v[i] = v0[i];
      b2_rounds_wide<10, 1>(v, m);
#pragma unroll
      for (int i = 0; i < 4; i++) h[i] = h0[i] ^ v[i] ^ v[8 + i];
      tz = digest_trailing_zeros<M31_OUT>(h);
    } else {
      tz = pow_trailing_zeros<M31_OUT>(prefix, nonce);
    }
    uint64_t hit = ~0ull;
    if (n < end && tz >= bits) hit = n;
    hit = wave_min_u64(hit);
    if ((threadIdx.x & 63) == 0 && hit != ~0ull) atomicMin(best, (unsigned long long)hit);
  }
}

// 512 workgroups of 256 lanes are two wavefronts per SIMD of 256 CUs.
template <bool STWO>
static void launch_grind(uint32_t grid, bool m31_out, const uint32_t* prefix, uint32_t bits, unsigned long long* best,
                         uint64_t start, uint64_t count, hipStream_t s) {
  const bool wide = grid >= 512;
  hipLaunchKernelGGL(m31_out ? (wide ? k_grind<STWO, true, true> : k_grind<STWO, true, false>)
                             : (wide ? k_grind<STWO, false, true> : k_grind<STWO, false, false>),
                     dim3(grid), dim3(256), 0, s, prefix, bits, best, start, count);
  VX_HIP(hipGetLastError());
}

__global__ void k_set_u64(unsigned long long* p, unsigned long long v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}
__global__ void k_stwo_index_to_nonce(unsigned long long* p) {
  if (threadIdx.x == 0 && blockIdx.x == 0 && *p != ~0ull) *p = stwo_nonce(*p);
}

// Workgroups of a search for `bits` trailing zeros. Every lane of the grid
// tests one nonce per round until the round passes the smallest hit, so a
// search tests about (hit + one round of the grid) nonces; a round of a
// quarter of the expected 2^bits nonces keeps that overshoot small (PoW 20:
// 1024 workgroups, 2^18 lanes), and large searches use the whole GPU
// (2048 workgroups, 8 per CU).
static uint32_t grind_grid(uint32_t bits) {
  const uint64_t wgs = bits >= 20 + 1 ? 2048ull : (1ull << bits) / 4 / 256;
  return (uint32_t)(wgs < 64 ? 64 : (wgs > 2048 ? 2048 : wgs));
}

// Whole search over the stwo family: the same increasing-index scan, then
// the winning index is turned into its nonce. Indices up to 2^44 cover
// hi < 2^24.
// m31_out selects the Blake2sChannelGeneric<true> test (output words
// reduced mod P before the trailing-zero count).
void grind_pow_stwo(const uint32_t* d_prefix, uint32_t pow_bits, uint64_t* d_result, bool m31_out, hipStream_t s) {
  require(pow_bits >= 1 && pow_bits <= 32, "grind_pow_stwo: pow_bits must be 1..32");
  auto* best = reinterpret_cast<unsigned long long*>(d_result);
  hipLaunchKernelGGL(k_set_u64, dim3(1), dim3(64), 0, s, best, ~0ull);
  launch_grind<true>(grind_grid(pow_bits), m31_out, d_prefix, pow_bits, best, 0ull, GRIND_LIMIT, s);
  hipLaunchKernelGGL(k_stwo_index_to_nonce, dim3(1), dim3(64), 0, s, best);
  VX_HIP(hipGetLastError());
}

// `preset`: *d_result is ~0 already.
void grind_pow(const uint32_t* d_prefix, uint32_t pow_bits, uint64_t* d_result, hipStream_t s, bool preset) {
  require(pow_bits >= 1 && pow_bits <= 32, "grind_pow: pow_bits must be 1..32");
  auto* best = reinterpret_cast<unsigned long long*>(d_result);
  if (!preset) hipLaunchKernelGGL(k_set_u64, dim3(1), dim3(64), 0, s, best, ~0ull);
  // every lane loops until its nonce exceeds the best hit
  launch_grind<false>(grind_grid(pow_bits), false, d_prefix, pow_bits, best, 0ull, GRIND_LIMIT, s);
}

// Reference-style batch (cuda/grind.cu:94-110): test nonces
// [batch_offset, batch_offset + n) and atomicMin hits into *d_result.
void grind_pow_batch(const uint32_t* d_prefix, uint64_t* d_result, uint32_t pow_bits, uint64_t batch_offset,
                     uint64_t n, bool m31_out, hipStream_t s) {
  require(pow_bits <= 128 && n > 0, "grind_pow_batch: bad arguments");
  uint64_t blocks = (n + 255) / 256;
  uint32_t grid = (uint32_t)(blocks < 4096 ? blocks : 4096);
  auto* best = reinterpret_cast<unsigned long long*>(d_result);
  launch_grind<false>(grid, m31_out, d_prefix, pow_bits, best, batch_offset, n, s);
}

__global__ void k_write_words(uint32_t* dst, WordWrites w) {
  if (threadIdx.x < w.n) dst[w.at[threadIdx.x]] = w.value[threadIdx.x];
}

// A few words at scattered places by one launch.
void write_words(uint32_t* dst, const WordWrites& w, hipStream_t s) {
  if (w.n == 0) return;
  hipLaunchKernelGGL(k_write_words, dim3(1), dim3(64), 0, s, dst, w);
  VX_HIP(hipGetLastError());
}

// Proof download by the GPU itself: the workgroups store the proof
// straight into pinned host memory (mapped into the device's address space),
// 16 bytes per lane per step, instead of a DMA copy whose start-up cost
// dominated for 1-2 MB proofs.
// The destination is read from device memory (set_inputs), so that the copy
// belongs to the proof's captured graph.
__global__ __launch_bounds__(256) void k_copy_to_host(uint32_t* const* dst_p, const uint32_t* src, uint64_t words) {
  uint32_t* const dst = *dst_p;
  const uint64_t n16 = words >> 2;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  uint4* d4 = reinterpret_cast<uint4*>(dst);
  const uint4* s4 = reinterpret_cast<const uint4*>(src);
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) d4[i] = s4[i];
  const uint64_t tail = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tail < (words & 3)) dst[4 * n16 + tail] = src[4 * n16 + tail];
}

void copy_to_host(uint32_t* const* d_dst, const uint32_t* dev_src, uint64_t words, hipStream_t s) {
  require((reinterpret_cast<uintptr_t>(dev_src) & 15u) == 0, "copy_to_host: 16-byte aligned source");
  const uint64_t blocks = ((words >> 2) + 255) / 256;
  const uint32_t grid = (uint32_t)(blocks < 1 ? 1 : (blocks > 512 ? 512 : blocks));
  hipLaunchKernelGGL(k_copy_to_host, dim3(grid), dim3(256), 0, s, d_dst, dev_src, words);
  VX_HIP(hipGetLastError());
}

}  // namespace vx
