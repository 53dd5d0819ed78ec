// Evaluation of stwo-basis polynomials at a QM31 point, and barycentric sums
// (the stwo plugin's PolyOps::eval_at_point / barycentric_eval_at_point).
//
// Semantics: f(z) = sum_i c_i prod_{bit b of i} F[b] with F[b] =
// factors[log_n - 1 - b]: factors[0] folds the top coefficient bit
// (cuda/circle_ntt.cu:186-231, 429-468; the plugin passes the mappings
// [y, x, pi(x), ...] reversed, crates/cuda-backend/src/poly_ops.rs:382-443).
// All arithmetic is exact, so any summation order gives the same value.
//
// MI355X design: the reference folds level by level (log_n launches, each
// reading and writing a QM31 vector, 16 bytes per element at the first
// level). Here the M31 coefficients are read once, by k_eval_big (n >= 2^14:
// 64 coefficients per lane, coalesced loads, the basis as scalars) or
// k_eval_blocks (smaller n: 16 consecutive coefficients per lane against the
// 16 products of F[0..3] in LDS). Products are accumulated 4 per 64-bit sum
// before a reduction; a workgroup folds its lanes in LDS, and the block sums
// are folded 256 at a time with the next 8 factors.
#include <algorithm>

#include "prover.h"
#include "vx_internal.h"
#include "vx_blake2s_x4.h"

namespace vx {

static constexpr uint32_t EV_LANE_LOG = 4;   // coefficients per lane: 16
static constexpr uint32_t EV_WG = 256;       // lanes per workgroup
static constexpr uint32_t EV_WG_LOG = 8;

__device__ __forceinline__ qm31 ld_factor(const uint32_t* factors, uint32_t log_n, uint32_t b) {
  return ld_uniform(reinterpret_cast<const qm31*>(factors) + (log_n - 1 - b));
}

// Folds q[0..W) (W = blockDim.x, a power of two) in LDS with F[fb + j] for
// level j: q[t] += F[fb + j] * q[t + 2^j]. Returns q[0] (valid in lane 0).
__device__ qm31 lds_fold(qm31* q, qm31 v, const uint32_t* factors, uint32_t log_n, uint32_t fb) {
  const uint32_t t = threadIdx.x, W = blockDim.x;
  q[t] = v;
  __syncthreads();
  for (uint32_t j = 0; (1u << j) < W; j++) {
    const qm31 f = ld_factor(factors, log_n, fb + j);
    if ((t & ((2u << j) - 1)) == 0) q[t] = qm_add(q[t], qm_mul(f, q[t + (1u << j)]));
    __syncthreads();
  }
  return q[0];
}

// Block sums of 16 * blockDim.x coefficients each.
__global__ __launch_bounds__(EV_WG) void k_eval_blocks(const uint32_t* __restrict__ c, const uint32_t* factors,
                                                       uint32_t log_n, uint32_t* __restrict__ part) {
  __shared__ qm31 basis[16];
  __shared__ qm31 q[EV_WG];
  const uint32_t t = threadIdx.x;
  for (uint32_t m = t; m < 16; m += blockDim.x) {
    qm31 b{{1u, 0u, 0u, 0u}};
    for (uint32_t k = 0; k < EV_LANE_LOG; k++)
      if ((m >> k) & 1u) b = qm_mul(b, ld_factor(factors, log_n, k));
    basis[m] = b;
  }
  const uint64_t g = (uint64_t)blockIdx.x * blockDim.x + t;
  const uint4* p = reinterpret_cast<const uint4*>(c + (g << EV_LANE_LOG));
  uint32_t cv[16];
#pragma unroll
  for (uint32_t m = 0; m < 4; m++) {
    const uint4 x = p[m];
    cv[4 * m] = x.x;
    cv[4 * m + 1] = x.y;
    cv[4 * m + 2] = x.z;
    cv[4 * m + 3] = x.w;
  }
  __syncthreads();
  qm31 s;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) {
    uint32_t r = 0;
#pragma unroll
    for (uint32_t grp = 0; grp < 4; grp++) {
      uint64_t acc = 0;  // 4 products < 4 P^2 < 2^64
#pragma unroll
      for (uint32_t m = 0; m < 4; m++) acc += (uint64_t)cv[4 * grp + m] * basis[4 * grp + m].v[k];
      r = m31_add(r, m31_reduce64(acc));
    }
    s.v[k] = r;
  }
  const qm31 v = lds_fold(q, s, factors, log_n, EV_LANE_LOG);
  if (t == 0) reinterpret_cast<qm31*>(part)[blockIdx.x] = v;
}

// Folds blockDim.x consecutive QM31 sums (covering coefficient bits from fb up).
__global__ __launch_bounds__(EV_WG) void k_eval_tree(const uint32_t* __restrict__ in, const uint32_t* factors,
                                                     uint32_t log_n, uint32_t fb, uint32_t* __restrict__ out) {
  __shared__ qm31 q[EV_WG];
  const qm31 v = reinterpret_cast<const qm31*>(in)[(uint64_t)blockIdx.x * blockDim.x + threadIdx.x];
  const qm31 r = lds_fold(q, v, factors, log_n, fb);
  if (threadIdx.x == 0) reinterpret_cast<qm31*>(out)[blockIdx.x] = r;
}

// ---- n >= 2^14: 64 coefficients per lane, basis in scalar registers.
// A workgroup covers 2^14 coefficients. Lane t reads the 16 uint4 at
// t + 256 m (m < 16), fully coalesced, so coefficient r + 4t + 1024m sits in
// component r of load m: bits 0-1 = r, 2-9 = t, 10-13 = m. The setup kernel
// tabulates E[r + 4 m01] = prod of F[0], F[1], F[10], F[11] over the set
// bits of (r, m01) and D[m23] over F[12], F[13]; lanes read them as
// wave-uniform scalars. Per lane: four 16-term sums w[m23] against E, then
// w0 + D1 w1 + D2 w2 + D3 w3; the 256 lanes are folded with F[2..9].
// (Per 2^14 coefficients a wave issues about 1600 VALU instructions, a
// quarter of the 16-per-lane kernel's; at 2^24 this kernel takes 27 us
// against 50 us. Looping each workgroup over several chunks with the next
// chunk's loads in flight measured the same 27 us.)
static constexpr uint32_t EV_BIG_LOG = 14;

__global__ void k_eval_setup(const uint32_t* factors, uint32_t log_n, uint32_t* table) {
  const uint32_t q = threadIdx.x;  // 0..15: E[q]; 16..19: D[q - 16]
  qm31 b{{1u, 0u, 0u, 0u}};
  if (q < 16) {
    const uint32_t bits[4] = {0, 1, 10, 11};
    for (uint32_t k = 0; k < 4; k++)
      if ((q >> k) & 1u) b = qm_mul(b, ld_factor(factors, log_n, bits[k]));
  } else if (q < 20) {
    for (uint32_t k = 0; k < 2; k++)
      if (((q - 16) >> k) & 1u) b = qm_mul(b, ld_factor(factors, log_n, 12 + k));
  }
  if (q < 20) reinterpret_cast<qm31*>(table)[q] = b;
}

__global__ __launch_bounds__(EV_WG) void k_eval_big(const uint32_t* __restrict__ c, const uint32_t* table,
                                                    const uint32_t* factors, uint32_t log_n,
                                                    uint32_t* __restrict__ part) {
  __shared__ qm31 q[EV_WG];
  const uint32_t t = threadIdx.x;
  const uint4* p = reinterpret_cast<const uint4*>(c) + ((uint64_t)blockIdx.x << (EV_BIG_LOG - 2)) + t;
  uint4 x[16];
#pragma unroll
  for (uint32_t m = 0; m < 16; m++) x[m] = p[m * EV_WG];
  uniform_t<qm31>* E = (uniform_t<qm31>*)table;
  qm31 w[4];
#pragma unroll
  for (uint32_t m23 = 0; m23 < 4; m23++) {
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
      uint32_t r = 0;
#pragma unroll
      for (uint32_t m01 = 0; m01 < 4; m01++) {
        const uint4 v = x[m01 + 4 * m23];
        // 4 products < 4 P^2 < 2^64
        const uint64_t acc = (uint64_t)v.x * E[4 * m01].v[k] + (uint64_t)v.y * E[4 * m01 + 1].v[k] +
                             (uint64_t)v.z * E[4 * m01 + 2].v[k] + (uint64_t)v.w * E[4 * m01 + 3].v[k];
        r = m31_add(r, m31_reduce64(acc));
      }
      w[m23].v[k] = r;
    }
  }
  qm31 v = w[0];
#pragma unroll
  for (uint32_t m23 = 1; m23 < 4; m23++)
    v = qm_add(v, qm_mul(ld_uniform(reinterpret_cast<const qm31*>(table) + 16 + m23), w[m23]));
  const qm31 s = lds_fold(q, v, factors, log_n, 2);
  if (t == 0) reinterpret_cast<qm31*>(part)[blockIdx.x] = s;
}

// n < 16: one lane.
__global__ void k_eval_small(const uint32_t* c, const uint32_t* factors, uint32_t log_n, uint32_t* out) {
  qm31 v[8];
  const uint32_t n = 1u << log_n;
  if (log_n == 0) {
    reinterpret_cast<qm31*>(out)[0] = qm31{{c[0], 0u, 0u, 0u}};
    return;
  }
  const qm31 f0 = ld_factor(factors, log_n, 0);
  for (uint32_t i = 0; i < n / 2; i++) v[i] = qm_add(qm31{{c[2 * i], 0u, 0u, 0u}}, qm_scale(f0, c[2 * i + 1]));
  for (uint32_t b = 1, m = n / 2; m > 1; b++, m >>= 1) {
    const qm31 f = ld_factor(factors, log_n, b);
    for (uint32_t i = 0; i < m / 2; i++) v[i] = qm_add(v[2 * i], qm_mul(f, v[2 * i + 1]));
  }
  reinterpret_cast<qm31*>(out)[0] = v[0];
}

const uint32_t* eval_at_point(const uint32_t* c, const uint32_t* factors, uint32_t log_n, uint32_t* s1,
                              uint32_t* s2, hipStream_t s) {
  require(log_n <= 31, "eval_at_point: log_n must be <= 31");
  if (log_n < EV_LANE_LOG) {
    hipLaunchKernelGGL(k_eval_small, dim3(1), dim3(1), 0, s, c, factors, log_n, s1);
    VX_HIP(hipGetLastError());
    return s1;
  }
  uint32_t groups_log, fb;
  uint32_t* in = s1;
  uint32_t* out = s2;
  if (log_n >= EV_BIG_LOG) {
    // the 20-entry table sits in s2 until the first tree level overwrites it
    hipLaunchKernelGGL(k_eval_setup, dim3(1), dim3(64), 0, s, factors, log_n, s2);
    VX_HIP(hipGetLastError());
    groups_log = log_n - EV_BIG_LOG;
    hipLaunchKernelGGL(k_eval_big, dim3(1u << groups_log), dim3(EV_WG), 0, s, c, s2, factors, log_n, s1);
    VX_HIP(hipGetLastError());
    fb = EV_BIG_LOG;
  } else {
    const uint32_t lanes_log = log_n - EV_LANE_LOG;
    const uint32_t wg_log = lanes_log < EV_WG_LOG ? lanes_log : EV_WG_LOG;
    groups_log = lanes_log - wg_log;
    hipLaunchKernelGGL(k_eval_blocks, dim3(1u << groups_log), dim3(1u << wg_log), 0, s, c, factors, log_n, s1);
    VX_HIP(hipGetLastError());
    fb = EV_LANE_LOG + wg_log;
  }
  while (groups_log > 0) {
    const uint32_t w = groups_log < EV_WG_LOG ? groups_log : EV_WG_LOG;
    groups_log -= w;
    hipLaunchKernelGGL(k_eval_tree, dim3(1u << groups_log), dim3(1u << w), 0, s, in, factors, log_n, fb, out);
    VX_HIP(hipGetLastError());
    fb += w;
    uint32_t* tmp = in;
    in = out;
    out = tmp;
  }
  return in;
}

// ---------------------------------------------------------------------------
// Many columns at one or two points (the OODS step evaluates every committed
// column at z and at z_next; cuda/batch_eval_at_point.cu:11-100 restricts
// this to n <= 64). A column of 2^L coefficients uses the last L of the
// max_log_n factors, so coefficient bit b of every column is folded by the
// same F[b] = factors[max_log_n - 1 - b], and the weight of a coefficient is
// a product over its index bits. Columns are cut into chunks of 2^14
// coefficients (shorter columns are one chunk, the words past their end read
// as zero); in a chunk lane t reads the 16 uint4 at t + 256 m, so index bits
// 0-1 are the component r, 2-9 the lane, 10-13 m, and from 14 up the chunk:
//   f(z) = sum_chunk G[chunk] sum_t L[t] sum_j E[j] c,  j = (r, m), 64 values.
// The tables E, L and G are made once per call (k_eval_tables). A workgroup
// takes some consecutive chunks of a column: per chunk each lane forms its
// 64-term sums against E (wave-uniform scalars) and adds G[chunk] times them
// to its own; L[t] and the sum over the lanes follow once at the end, and a
// second launch adds the workgroups' sums.
//
// Bound by the read of the columns once the arithmetic is small: a term is
// one multiply-add per component into a signed 64-bit sum (weights centred to
// |w| < 2^30, coefficients shifted by 2^30, so eight products fit before a
// fold; the shift's share of the sum is the constant C). The tree folds of
// the lanes by QM31 products that this replaces were two thirds of the
// kernel's instructions. 64 columns of 2^20 at two points (268 MB): 192 -> 51 us
// (the read at a large copy's rate takes 52); the OODS step 338 -> 117 us.
static constexpr uint32_t EV_TERMS = 64;      // coefficients per lane and chunk
static constexpr uint32_t EV_MAX_WGS = 2048;  // of a call: chunks per workgroup grow beyond
static constexpr uint32_t EV_ARG_COLS = 192;  // columns that travel in the kernels' arguments

struct EvalCol {
  const uint32_t* p;
  uint32_t first;  // workgroup of the column's first chunk, ascending from 0
  uint32_t log_n;
};
// The columns are an array in the kernels' own arguments, or, when there are
// more, a table uploaded into the workspace. (Splitting them over launches of
// EV_ARG_COLS columns instead took 676 us for 10,000 columns of 2^8, the table
// takes 114; 500 columns 52 and 33.)
struct EvalArgs {
  EvalCol col[EV_ARG_COLS];
};
__device__ __forceinline__ EvalCol eval_col(const EvalArgs& cols, uint32_t k) { return cols.col[k]; }
__device__ __forceinline__ EvalCol eval_col(const EvalCol* cols, uint32_t k) { return ld_uniform(cols + k); }
// words of the tables of np points, G having 2^g_log entries
struct EvalTables {
  uint32_t np, g_log;
  __host__ __device__ uint64_t e() const { return 0; }                              // [64][np] centred QM31
  __host__ __device__ uint64_t c() const { return 4ull * EV_TERMS * np; }           // [np]
  __host__ __device__ uint64_t l() const { return c() + 4ull * np; }                // [np][256]
  __host__ __device__ uint64_t g() const { return l() + 4ull * EV_WG * np; }        // [np][2^g_log]
  __host__ __device__ uint64_t words() const { return g() + (4ull * np << g_log); }
};

__device__ __forceinline__ qm31 factor_or_one(const uint32_t* factors, uint32_t max_log_n, uint32_t b) {
  return b < max_log_n ? ld_factor(factors, max_log_n, b) : qm31{{1u, 0u, 0u, 0u}};
}

// One entry per lane; blockIdx.y = point.
__global__ __launch_bounds__(EV_WG) void k_eval_tables(const uint32_t* factors, uint32_t max_log_n, EvalTables T,
                                                       uint32_t* tables) {
  const uint32_t pt = blockIdx.y;
  uint32_t x = blockIdx.x * EV_WG + threadIdx.x;
  factors += (uint64_t)pt * 4 * (max_log_n ? max_log_n : 1);
  qm31* out = reinterpret_cast<qm31*>(tables);
  const qm31 one{{1u, 0u, 0u, 0u}};
  qm31 b = one;
  if (x <= EV_TERMS) {  // E[x], or C = 2^30 times their sum, the product of 1 + F over the bits
#pragma unroll
    for (uint32_t k = 0; k < 6; k++) {
      const qm31 f = factor_or_one(factors, max_log_n, k < 2 ? k : 8 + k);
      if (x == EV_TERMS) b = qm_mul(b, qm_add(one, f));
      else if ((x >> k) & 1u) b = qm_mul(b, f);
    }
    if (x == EV_TERMS) {
      out[T.c() / 4 + pt] = qm_scale(b, 1u << 30);
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) b.v[k] = b.v[k] > P / 2 ? b.v[k] - P : b.v[k];
      out[T.e() / 4 + x * T.np + pt] = b;
    }
    return;
  }
  x -= EV_TERMS + 1;
  if (x < EV_WG) {
#pragma unroll
    for (uint32_t k = 0; k < EV_WG_LOG; k++)
      if ((x >> k) & 1u) b = qm_mul(b, factor_or_one(factors, max_log_n, 2 + k));
    out[T.l() / 4 + pt * EV_WG + x] = b;
    return;
  }
  x -= EV_WG;
  if (x >> T.g_log) return;
  for (uint32_t k = 0; k < T.g_log; k++)
    if ((x >> k) & 1u) b = qm_mul(b, ld_factor(factors, max_log_n, EV_BIG_LOG + k));
  out[T.g() / 4 + ((uint64_t)pt << T.g_log) + x] = b;
}

// lo + 2 hi, congruent mod P: below 2^33 in absolute value for any x. One
// v_mad_i64_i32 (see m31_fold64).
__device__ __forceinline__ int64_t fold_signed(int64_t x) {
  int32_t two = 2;
  asm("" : "+s"(two));
  return (int64_t)(int32_t)(x >> 32) * two + (uint32_t)x;
}
__device__ __forceinline__ uint32_t wave_sum_mod_p(uint32_t v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = m31_add(v, (uint32_t)__shfl_xor((int)v, off, 64));
  return v;
}

// A workgroup takes 2^cpw_log chunks.
template <uint32_t NP, typename Cols>
__global__ __launch_bounds__(EV_WG) void k_eval_chunks(Cols cols, uint32_t n_cols, uint32_t cpw_log, EvalTables T,
                                                       const uint32_t* tables, uint32_t* part, uint32_t part_stride) {
  __shared__ qm31 red[NP][EV_WG / 64];
  const uint32_t wg = blockIdx.x, t = threadIdx.x;
  uint32_t lo = 0, hi = n_cols;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (eval_col(cols, mid).first <= wg) lo = mid;
    else hi = mid;
  }
  const EvalCol c = eval_col(cols, lo);
  const uint32_t* col = c.p;
  const uint32_t L = c.log_n;
  const uint32_t n = 1u << L;
  const uint32_t chunks = L > EV_BIG_LOG ? 1u << (L - EV_BIG_LOG) : 1u;
  const uint32_t c0 = (wg - c.first) << cpw_log, c1 = min(c0 + (1u << cpw_log), chunks);
  qm31 sum[NP];
#pragma unroll
  for (uint32_t pt = 0; pt < NP; pt++) sum[pt] = qm31{{0u, 0u, 0u, 0u}};
#pragma unroll 1
  for (uint32_t chunk = c0; chunk < c1; chunk++) {
    // load m of this lane: words w, w + 1, ... of the column (zero past its end)
    auto load = [&](uint32_t m) {
      const uint32_t w = 4 * (t + m * EV_WG);
      if (L >= EV_BIG_LOG) return *reinterpret_cast<const uint4*>(col + ((uint64_t)chunk << EV_BIG_LOG) + w);
      if (L >= 2) return w < n ? *reinterpret_cast<const uint4*>(col + w) : make_uint4(0u, 0u, 0u, 0u);
      return make_uint4(w < n ? col[w] : 0u, w + 1 < n ? col[w + 1] : 0u, 0u, 0u);
    };
    int64_t acc[NP][4];
#pragma unroll
    for (uint32_t pt = 0; pt < NP; pt++)
#pragma unroll
      for (int k = 0; k < 4; k++) acc[pt][k] = 0;
    uniform_t<int32_t>* E = (uniform_t<int32_t>*)(tables + T.e());
    uint4 x[2] = {load(0), load(1)};
    // A loop, not unrolled: the weights of a step fill 64 scalar registers, and
    // unrolled the compiler reads those of all steps ahead and spills them.
#pragma unroll 1
    for (uint32_t m = 0; m < 16; m += 2) {
      const uint4 y[2] = {x[0], x[1]};
      if (m < 14) {
        x[0] = load(m + 2);
        x[1] = load(m + 3);
      }
#pragma unroll
      for (uint32_t h = 0; h < 2; h++) {
        const uint32_t xv[4] = {y[h].x, y[h].y, y[h].z, y[h].w};
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) {
          const int64_t xs = (int32_t)(xv[r] - (1u << 30));
#pragma unroll
          for (uint32_t pt = 0; pt < NP; pt++)
#pragma unroll
            for (int k = 0; k < 4; k++) acc[pt][k] += xs * E[4 * (NP * (4 * h + r) + pt) + k];
        }
      }
      E += 4 * NP * 8;
      // eight products of at most 2^30 (2^30 - 1) and a folded sum stay below 2^63
#pragma unroll
      for (uint32_t pt = 0; pt < NP; pt++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[pt][k] = fold_signed(acc[pt][k]);
    }
#pragma unroll
    for (uint32_t pt = 0; pt < NP; pt++) {
      const qm31 C = ld_uniform(reinterpret_cast<const qm31*>(tables + T.c()) + pt);
      qm31 s;
#pragma unroll
      for (int k = 0; k < 4; k++) s.v[k] = m31_reduce64((uint64_t)(acc[pt][k] + ((int64_t)P << 3)) + C.v[k]);
      if (chunk != 0) {  // G[0] = 1
        const qm31_mat g =
            qm_left_matrix(ld_uniform(reinterpret_cast<const qm31*>(tables + T.g()) + ((uint64_t)pt << T.g_log) + chunk));
        qm31 r;
#pragma unroll
        for (int k = 0; k < 4; k++)
          r.v[k] = m31_reduce64((uint64_t)g.m[k][0] * s.v[0] + (uint64_t)g.m[k][1] * s.v[1] +
                                (uint64_t)g.m[k][2] * s.v[2] + (uint64_t)g.m[k][3] * s.v[3]);
        s = r;
      }
      sum[pt] = qm_add(sum[pt], s);
    }
  }
#pragma unroll
  for (uint32_t pt = 0; pt < NP; pt++) {
    const uint4 lv = reinterpret_cast<const uint4*>(tables + T.l())[pt * EV_WG + t];
    qm31 s = qm_mul_lazy(qm31{{lv.x, lv.y, lv.z, lv.w}}, sum[pt]);
#pragma unroll
    for (int k = 0; k < 4; k++) s.v[k] = wave_sum_mod_p(s.v[k]);
    if ((t & 63) == 0) red[pt][t >> 6] = s;
  }
  __syncthreads();
  if (t < NP) {
    qm31 s = red[t][0];
    for (uint32_t w = 1; w < EV_WG / 64; w++) s = qm_add(s, red[t][w]);
    reinterpret_cast<qm31*>(part)[(uint64_t)t * part_stride + wg] = s;
  }
}

// results[pt * n_cols + k] = the sum of column k's workgroups' sums; one
// wavefront per (column, point).
template <typename Cols>
__global__ __launch_bounds__(64) void k_eval_sum(Cols cols, uint32_t n_cols, uint32_t n_wgs, const uint32_t* part,
                                                 uint32_t* results) {
  const uint32_t k = blockIdx.x, pt = blockIdx.y, lane = threadIdx.x;
  const uint32_t b = eval_col(cols, k).first, e = k + 1 < n_cols ? eval_col(cols, k + 1).first : n_wgs;
  const qm31* p = reinterpret_cast<const qm31*>(part) + (uint64_t)pt * n_wgs;
  uint64_t s[4] = {0, 0, 0, 0};
  for (uint32_t i = b + lane; i < e; i += 64)
#pragma unroll
    for (int c = 0; c < 4; c++) s[c] += p[i].v[c];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const uint32_t v = wave_sum_mod_p(m31_reduce64(s[c]));
    if (lane == 0) results[4 * ((uint64_t)pt * n_cols + k) + c] = v;
  }
}

// The split of a batch into workgroups and its workspace, after checking it.
struct EvalPlan {
  EvalTables T{};
  uint32_t cpw_log = 0;
  uint32_t wgs = 0;
  std::vector<EvalCol> cols;
  uint64_t part_words() const { return 4ull * T.np * wgs; }
  uint64_t col_words() const { return cols.size() > EV_ARG_COLS ? cols.size() * (sizeof(EvalCol) / 4) : 0; }
  uint64_t ws_words() const { return T.words() + part_words() + col_words(); }
};
static uint32_t eval_wgs_of(uint32_t L, uint32_t cpw_log) {
  const uint32_t c = L > EV_BIG_LOG ? L - EV_BIG_LOG : 0;
  return c > cpw_log ? 1u << (c - cpw_log) : 1u;
}
static EvalPlan eval_plan(const uint32_t* const* h_cols, const uint32_t* h_log_sizes, uint32_t n_cols, uint32_t np,
                          uint32_t max_log_n) {
  require(np == 1 || np == 2, "eval_at_point_batch: one or two points");
  require(max_log_n <= 31, "eval_at_point_batch: max_log_n must be <= 31");
  uint64_t total = 0;
  uint32_t top = 0;
  for (uint32_t k = 0; k < n_cols; k++) {
    const uint32_t L = h_log_sizes[k];
    require(h_cols[k] != nullptr && L <= max_log_n, "eval_at_point_batch: null column or log size above max_log_n");
    require(L < 2 || (reinterpret_cast<uintptr_t>(h_cols[k]) & 15u) == 0,
            "eval_at_point_batch: columns must be 16-byte aligned");
    total += L > EV_BIG_LOG ? 1ull << (L - EV_BIG_LOG) : 1ull;
    top = L > top ? L : top;
  }
  require(total < (1ull << 31), "eval_at_point_batch: too many chunks");
  // Chunks per workgroup: the lanes' products by L and their sum are paid
  // once per workgroup, so no more workgroups than keep the chip full.
  uint32_t cpw_log = 0;
  while ((total >> cpw_log) > EV_MAX_WGS) cpw_log++;
  EvalPlan plan;
  plan.T = EvalTables{np, top > EV_BIG_LOG ? top - EV_BIG_LOG : 0};
  plan.cpw_log = cpw_log;
  plan.cols.resize(n_cols);
  for (uint32_t k = 0; k < n_cols; k++) {
    plan.cols[k] = {h_cols[k], plan.wgs, h_log_sizes[k]};
    plan.wgs += eval_wgs_of(h_log_sizes[k], cpw_log);
  }
  return plan;
}

template <typename Cols>
static void eval_launch(const EvalPlan& plan, const Cols& cols, const uint32_t* tables, uint32_t* part,
                        uint32_t* results, hipStream_t s) {
  const uint32_t n = (uint32_t)plan.cols.size();
  hipLaunchKernelGGL((plan.T.np == 2 ? k_eval_chunks<2, Cols> : k_eval_chunks<1, Cols>), dim3(plan.wgs), dim3(EV_WG), 0,
                     s, cols, n, plan.cpw_log, plan.T, tables, part, plan.wgs);
  VX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_eval_sum<Cols>, dim3(n, plan.T.np), dim3(64), 0, s, cols, n, plan.wgs, part, results);
  VX_HIP(hipGetLastError());
}

// np points (1 or 2): factors holds np tables of 4 max_log_n words back to
// back (4 words when max_log_n is 0), results np arrays of n_cols QM31. The
// work is enqueued on s; the plan and the workspace (ws_words) must outlive it.
static void eval_batch_points(const EvalPlan& plan, const uint32_t* factors, uint32_t max_log_n, uint32_t* results,
                              uint32_t* ws, hipStream_t s) {
  const EvalTables& T = plan.T;
  const uint32_t n_cols = (uint32_t)plan.cols.size();
  uint32_t* tables = ws;
  uint32_t* part = tables + T.words();
  const uint64_t entries = EV_TERMS + 1 + EV_WG + (1ull << T.g_log);
  hipLaunchKernelGGL(k_eval_tables, dim3((uint32_t)((entries + EV_WG - 1) / EV_WG), T.np), dim3(EV_WG), 0, s, factors,
                     max_log_n, T, tables);
  VX_HIP(hipGetLastError());
  if (n_cols <= EV_ARG_COLS) {
    EvalArgs a{};
    std::copy(plan.cols.begin(), plan.cols.end(), a.col);
    eval_launch(plan, a, tables, part, results, s);
  } else {
    EvalCol* table = reinterpret_cast<EvalCol*>(part + plan.part_words());
    VX_HIP(hipMemcpyAsync(table, plan.cols.data(), sizeof(EvalCol) * n_cols, hipMemcpyHostToDevice, s));
    eval_launch(plan, static_cast<const EvalCol*>(table), tables, part, results, s);
  }
}

void eval_at_point_batch(const uint32_t* const* h_cols, const uint32_t* h_log_sizes, uint32_t n_cols,
                         const uint32_t* factors, uint32_t max_log_n, uint32_t* results, hipStream_t s) {
  if (n_cols == 0) return;
  const EvalPlan plan = eval_plan(h_cols, h_log_sizes, n_cols, 1, max_log_n);
  DeviceBuf ws(4 * plan.ws_words());
  eval_batch_points(plan, factors, max_log_n, results, ws.u32(), s);
  VX_HIP(hipStreamSynchronize(s));  // the workspace is freed on return
}

// ---------------------------------------------------------------------------
// Barycentric sum (cuda/barycentric_eval.cu:41-99): block b of n_blocks
// 256-lane blocks accumulates evals[i] * weights[i] (QM31 AoS) over the
// grid-stride set i = (b * 256 + t) + k * n_blocks * 256, and writes its
// partial sum out[4b..4b+4). Same partition as the reference, so every
// partial is the same value. Products are accumulated 4 per 64-bit sum.
static constexpr uint32_t BARY_THREADS = 256;

__global__ __launch_bounds__(BARY_THREADS) void k_barycentric(const uint32_t* __restrict__ ev,
                                                              const uint32_t* __restrict__ w, uint32_t n,
                                                              uint32_t* __restrict__ out) {
  __shared__ qm31 q[BARY_THREADS];
  const uint32_t t = threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * BARY_THREADS;
  uint32_t r[4] = {0u, 0u, 0u, 0u};
  uint64_t acc[4] = {0, 0, 0, 0};
  uint32_t pending = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * BARY_THREADS + t; i < n; i += stride) {
    const uint32_t e = ev[i];
    const uint4 x = reinterpret_cast<const uint4*>(w)[i];
    acc[0] += (uint64_t)e * x.x;
    acc[1] += (uint64_t)e * x.y;
    acc[2] += (uint64_t)e * x.z;
    acc[3] += (uint64_t)e * x.w;
    if (++pending == 4) {
      for (int k = 0; k < 4; k++) {
        r[k] = m31_add(r[k], m31_reduce64(acc[k]));
        acc[k] = 0;
      }
      pending = 0;
    }
  }
  for (int k = 0; k < 4; k++) r[k] = m31_add(r[k], m31_reduce64(acc[k]));
  q[t] = qm31{{r[0], r[1], r[2], r[3]}};
  __syncthreads();
  for (uint32_t h = BARY_THREADS / 2; h > 0; h >>= 1) {
    if (t < h) q[t] = qm_add(q[t], q[t + h]);
    __syncthreads();
  }
  if (t == 0) reinterpret_cast<qm31*>(out)[blockIdx.x] = q[0];
}

void barycentric_partials(const uint32_t* ev, const uint32_t* w, uint32_t n, uint32_t* out, uint32_t n_blocks,
                          hipStream_t s) {
  require(n_blocks >= 1 && n_blocks <= 65535, "barycentric: 1..65535 blocks");
  require((reinterpret_cast<uintptr_t>(w) & 15u) == 0, "barycentric: weights must be 16-byte aligned");
  hipLaunchKernelGGL(k_barycentric, dim3(n_blocks), dim3(BARY_THREADS), 0, s, ev, w, n, out);
  VX_HIP(hipGetLastError());
}

// ------------------------------------------------------------- OODS step
// src/oods.rs:44-81: t drawn from the channel, z = ((1 - t^2) / (1 + t^2),
// 2t / (1 + t^2)) on the QM31 circle, z_next = z * step with step the
// generator of the 2^trace_log subgroup (circle.rs generator doubled
// 31 - trace_log times); then both points' folding factors for max_log:
// [z.y, z.x, 2 z.x^2 - 1, ...] (max_log entries) reversed.
__device__ void oods_factors(qm31 zx, qm31 zy, uint32_t max_log, uint32_t* out) {
  qm31 x = zx;
  for (uint32_t i = 0; i < max_log; i++) {
    const qm31 m = i == 0 ? zy : x;
    if (i > 0) {
      const qm31 x2 = qm_mul_lazy(x, x);
      x = qm_sub(qm_add(x2, x2), qm31{{1u, 0u, 0u, 0u}});
    }
    for (int k = 0; k < 4; k++) out[4 * (max_log - 1 - i) + k] = m.v[k];
  }
}

// A dependent chain on one lane: the draw, the division, then max_log
// doublings. Lane 0 follows z and lane 1 z_next (both draw z), so the two
// chains of doublings run side by side: 22 -> 14 us for max_log 20.
__global__ void k_oods_point(uint32_t* ch_words, uint32_t trace_log, uint32_t max_log, uint32_t* points, uint32_t* fz,
                             uint32_t* fzn) {
  if (threadIdx.x > 1 || blockIdx.x != 0) return;
  const bool next = threadIdx.x == 1;
  Channel c;
  for (int i = 0; i < 8; i++) c.state[i] = ch_words[i];
  c.n_draws = ch_words[8];
  const qm31 t = ch_draw_felt(c);
  if (!next) {
    for (int i = 0; i < 8; i++) ch_words[i] = c.state[i];
    ch_words[8] = c.n_draws;
  }
  const qm31 one{{1u, 0u, 0u, 0u}};
  const qm31 t2 = qm_mul(t, t);
  const qm31 inv = qm_inv(qm_add(one, t2));
  const qm31 zx = qm_mul(qm_sub(one, t2), inv), zy = qm_mul(qm_add(t, t), inv);
  const cpt st = c_rdouble(c_generator(), 31 - trace_log);
  const qm31 nx = qm_sub(qm_scale(zx, st.x), qm_scale(zy, st.y));
  const qm31 ny = qm_add(qm_scale(zx, st.y), qm_scale(zy, st.x));
  const qm31 px = next ? nx : zx, py = next ? ny : zy;
  for (int k = 0; k < 4; k++) {
    points[(next ? 8 : 0) + k] = px.v[k];
    points[(next ? 12 : 4) + k] = py.v[k];
  }
  oods_factors(px, py, max_log, next ? fzn : fz);
}

// Channel::mix_felts (src/channel.rs:46-59) of the sampled values: the
// message is state || values; it is a dependent chain of compressions, which
// the four lanes of a quad share. All words are known beforehand, so the
// workgroup lays MIX_BLOCKS blocks at a time out in LDS in schedule order, one
// 16-byte read per round and lane, and one wavefront runs the chain over them
// with the next block's ten reads in flight: 300 instructions per lane and
// block instead of 430 with the words selected from registers. Bound by that
// chain: 64 columns (33 blocks) 36 -> 23 us, of which the layout is about 3.
static constexpr uint32_t MIX_BLOCKS = 64, MIX_THREADS = 640;
struct MixWords {
  uint8_t at[160];  // message word of schedule entry 16 round + 4 lane + k
};
constexpr MixWords make_mix_words() {
  MixWords t{};
  for (uint32_t e = 0; e < 160; e++) t.at[e] = (uint8_t)quad_word(e / 4 % 4, 4 * (e / 16) + e % 4);
  return t;
}
__constant__ const MixWords MIX_WORDS = make_mix_words();

__global__ __launch_bounds__(MIX_THREADS) void k_oods_mix(uint32_t* ch_words, const uint32_t* values,
                                                          uint32_t n_felts) {
  __shared__ uint32_t msg[16 * MIX_BLOCKS];
  __shared__ __align__(16) uint32_t sched[160 * MIX_BLOCKS];
  if (blockIdx.x != 0 || n_felts == 0) return;
  const uint32_t tid = threadIdx.x, q = tid & 3u, word = MIX_WORDS.at[tid % 160u];
  const bool q0 = q & 1, q1 = q & 2;
  uint32_t h_lo = sel4(q0, q1, VX_B2_IV0 ^ 0x01010020u, VX_B2_IV1, VX_B2_IV2, VX_B2_IV3);
  uint32_t h_hi = sel4(q0, q1, VX_B2_IV4, VX_B2_IV5, VX_B2_IV6, VX_B2_IV7);
  const uint64_t nwords = 8 + 4ull * n_felts;
  const uint32_t n_blocks = (uint32_t)((nwords + 15) / 16);
  for (uint32_t b0 = 0; b0 < n_blocks; b0 += MIX_BLOCKS) {
    const uint32_t nb = n_blocks - b0 < MIX_BLOCKS ? n_blocks - b0 : MIX_BLOCKS;
    __syncthreads();  // the chain is through with the blocks before
    for (uint32_t k = tid; k < 16 * nb; k += MIX_THREADS) {
      const uint64_t at = 16ull * b0 + k;
      msg[k] = at < 8 ? ch_words[at] : at < nwords ? values[at - 8] : 0u;
    }
    __syncthreads();
    for (uint32_t b = tid / 160u; b < nb; b += MIX_THREADS / 160u) sched[160 * b + tid % 160u] = msg[16 * b + word];
    __syncthreads();
    if (tid < 64) {
      const uint4* sq = reinterpret_cast<const uint4*>(sched) + q;
      auto read = [&](uint4 (&w)[10], uint32_t b) {
        // past the last block: the last one once more, unused
        const uint4* sn = sq + 40 * (b < nb ? b : nb - 1);
#pragma unroll
        for (int r = 0; r < 10; r++) w[r] = sn[4 * r];
        __builtin_amdgcn_sched_barrier(0);
      };
      auto compress = [&](const uint4 (&w)[10], uint32_t b) {
        const bool last = b0 + b + 1 == n_blocks;
        b2_compress_x4(h_lo, h_hi, w, last ? (uint32_t)(4 * nwords) : 64 * (b0 + b + 1), last, q);
      };
      uint4 w0[10], w1[10];  // taken in turn: no copies
      read(w0, 0);
      for (uint32_t b = 0; b < nb; b += 2) {
        read(w1, b + 1);
        compress(w0, b);
        if (b + 1 == nb) break;
        read(w0, b + 2);
        compress(w1, b + 1);
      }
    }
  }
  if (tid < 4) {
    ch_words[q] = h_lo;
    ch_words[4 + q] = h_hi;
  }
  if (tid == 0) ch_words[8] = 0;
}

void oods_sample(uint32_t* d_channel, const uint32_t* const* h_cols, const uint32_t* h_log_sizes, uint32_t n_cols,
                 uint32_t trace_log, uint32_t* d_points, uint32_t* d_values, hipStream_t s) {
  uint32_t max_log = 0;
  for (uint32_t k = 0; k < n_cols; k++) max_log = h_log_sizes[k] > max_log ? h_log_sizes[k] : max_log;
  const uint32_t fw = 4 * (max_log ? max_log : 1);
  // one allocation: both points' factors, then the evaluation's workspace
  EvalPlan plan;
  if (n_cols) plan = eval_plan(h_cols, h_log_sizes, n_cols, 2, max_log);
  const uint64_t ws_at = (2ull * fw + 63) & ~63ull;
  DeviceBuf buf(4 * (ws_at + (n_cols ? plan.ws_words() : 0)));
  uint32_t* fz = buf.u32();
  hipLaunchKernelGGL(k_oods_point, dim3(1), dim3(64), 0, s, d_channel, trace_log, max_log, d_points, fz, fz + fw);
  VX_HIP(hipGetLastError());
  if (n_cols) {
    // both points from one read of every column: values at z, then at z_next
    eval_batch_points(plan, fz, max_log, d_values, buf.u32() + ws_at, s);
    hipLaunchKernelGGL(k_oods_mix, dim3(1), dim3(MIX_THREADS), 0, s, d_channel, d_values, 2 * n_cols);
    VX_HIP(hipGetLastError());
  }
  VX_HIP(hipStreamSynchronize(s));  // the workspace is freed on return
}

}  // namespace vx
