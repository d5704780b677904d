// resident.hip -- set-up and host side of the resident conjugate gradients
// (resident_kernel.h): the pair layout of a matrix and the launch layout.
//
// Why one launch: with three kernels an iteration of a system that fits the
// caches is bound by launches and by the latencies at each kernel's start
// (state, partial sums, vectors from memory), about 5 us a kernel whatever it
// does; larger systems move every vector through memory 11 times an
// iteration.  Here an iteration is two barriers of 2-3 us and the matrix.
// FP64 Jacobi-PCG, MI355X, three kernels -> resident: 256 x 256 quads of two
// triangles (66049 rows) 16.3 -> 6.3 us an iteration; 48 x 52 x 45 nodes of
// tetrahedra numbered at random (112 thousand rows) 22 -> 11.3 us.  Mixed
// Jacobi-PCG on 128^3 hexes of six tetrahedra (2.15 million rows) to 1e-8
// 84.9 -> 34.8 ms; flexible PCG with a BF16 sparse preconditioner on 0.89
// million rows, assembly and inference included, 61.7 -> 24.7 ms.
#include "resident_kernel.h"

#include <algorithm>
#include <cmath>

namespace afem {
namespace resident {

// ---- pair layout --------------------------------------------------------------------------------
//
// One wave per slice.  The slice's rows are one contiguous range of the CSR
// arrays: it is read coalesced into LDS and each lane walks its row there
// (ranges that exceed the LDS space are walked in place).

constexpr int kStageMax = 4096; // entries of a slice staged in LDS

__device__ __forceinline__ void slice_rows(const int32_t* __restrict__ slice_row, int32_t nslice, int32_t s,
                                           const int32_t* __restrict__ rp, int lane, int32_t& row, bool& live,
                                           int32_t& b, int32_t& e, int32_t& e0, int32_t& e1)
{
  const int32_t r0 = slice_row[s], r1 = min(slice_row[2 * nslice + s], r0 + 64);
  row = r0 + lane;
  live = row < r1;
  e0 = rp[r0];
  e1 = rp[r1];
  b = live ? rp[row] : e1;
  e = live ? rp[row + 1] : e1;
}

// Pairs of every slice, and over the matrix: the longest row, the largest
// |column - row|, whether a non-empty row lacks its diagonal entry, whether a
// column leaves its row's segment, and the number of slices in most of whose
// entries neighbouring rows have unrelated columns.
__global__ void __launch_bounds__(64)
k_pair_count(int32_t nslice, const int32_t* __restrict__ slice_row, const int32_t* __restrict__ rp,
             const int32_t* __restrict__ ci, int32_t* __restrict__ width, int32_t* __restrict__ stats)
{
  __shared__ int32_t s_col[kStageMax];
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x;
  int32_t row, b, e, e0, e1;
  bool live;
  slice_rows(slice_row, nslice, s, rp, lane, row, live, b, e, e0, e1);
  const bool staged = e1 - e0 <= kStageMax;
  if (staged) {
    for (int32_t k = e0 + lane; k < e1; k += 64)
      s_col[k - e0] = ci[k];
    __syncthreads();
  }
  const int32_t g0 = slice_row[nslice + s], g1 = slice_row[2 * nslice + s];
  int32_t off = 0, far = 0, leaves = 0;
  for (int32_t k = b; k < e; ++k) {
    const int32_t c = staged ? s_col[k - e0] : ci[k];
    off += c != row ? 1 : 0;
    far = max(far, abs(c - row));
    leaves |= c < g0 || c >= g1 ? 2 : 0;
  }
  // entry j of this row against entry j of the row before: within a cache line or not
  const int32_t pb = __shfl_up(b, 1, 64), plen = __shfl_up(e, 1, 64) - pb;
  int32_t near = 0, both = lane > 0 && live ? min(e - b, plen) : 0;
  for (int32_t j = 0; j < both; ++j) {
    const int32_t c = staged ? s_col[b + j - e0] : ci[b + j], d = staged ? s_col[pb + j - e0] : ci[pb + j];
    near += abs(c - d) <= 8 ? 1 : 0;
  }
  int32_t pairs = (off + 1) / 2, len = e - b, lacks = ((e > b && off == e - b) ? 1 : 0) | leaves;
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    pairs = max(pairs, __shfl_xor(pairs, o, 64));
    len = max(len, __shfl_xor(len, o, 64));
    far = max(far, __shfl_xor(far, o, 64));
    lacks |= __shfl_xor(lacks, o, 64);
    near += __shfl_xor(near, o, 64);
    both += __shfl_xor(both, o, 64);
  }
  if (lane == 0) {
    width[s] = pairs;
    // a look first: almost every slice leaves the maxima as they are
    if (len > __hip_atomic_load(stats, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(stats, len);
    if (far > __hip_atomic_load(stats + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(stats + 1, far);
    if (lacks)
      atomicOr(stats + 2, lacks);
    if (2 * near < both)
      atomicAdd(stats + 3, 1);
  }
}

// ---- the same in another order of the rows ------------------------------------------------------
//
// Place i holds row perm[i], and its columns are places (inv).  A row's
// entries are taken in the order of their places, so that neighbouring rows
// read neighbouring elements; src keeps where they came from.

__global__ void k_invert(int32_t n, const int32_t* __restrict__ perm, int32_t* __restrict__ inv)
{
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    inv[perm[i]] = i;
}

__global__ void __launch_bounds__(64)
k_pairp_count(int32_t nslice, int32_t n, const int32_t* __restrict__ perm, const int32_t* __restrict__ inv,
              const int32_t* __restrict__ rp, const int32_t* __restrict__ ci, int32_t* __restrict__ width,
              int32_t* __restrict__ stats)
{
  const int32_t s = blockIdx.x;
  const int32_t i = s * 64 + threadIdx.x;
  const int32_t row = i < n ? perm[i] : -1;
  const int32_t b = row >= 0 ? rp[row] : 0, e = row >= 0 ? rp[row + 1] : 0;
  int32_t off = 0, far = 0;
  for (int32_t k = b; k < e; ++k) {
    const int32_t c = ci[k];
    off += c != row ? 1 : 0;
    far = max(far, abs(inv[c] - i));
  }
  int32_t pairs = (off + 1) / 2;
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    pairs = max(pairs, __shfl_xor(pairs, o, 64));
    far = max(far, __shfl_xor(far, o, 64));
  }
  if (threadIdx.x == 0) {
    width[s] = pairs;
    if (far > __hip_atomic_load(stats + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(stats + 1, far);
  }
}

template <class I>
__global__ void __launch_bounds__(64)
k_pairp_index(int32_t n, const int32_t* __restrict__ perm, const int32_t* __restrict__ inv,
              const int32_t* __restrict__ rp, const int32_t* __restrict__ ci, const int32_t* __restrict__ poff,
              I* __restrict__ idx, int32_t* __restrict__ src)
{
  typedef I I2 __attribute__((ext_vector_type(2)));
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x;
  const int32_t i = s * 64 + lane;
  const int32_t row = i < n ? perm[i] : -1;
  const int32_t b = row >= 0 ? rp[row] : 0, e = row >= 0 ? rp[row + 1] : 0;
  // (place, position) taken last: equal columns keep their CSR order
  int32_t place = -1, pos = -1;
  auto next = [&](int32_t& from) -> I {
    int32_t best = 0x7fffffff, at = -1;
    for (int32_t k = b; k < e; ++k) {
      const int32_t c = ci[k];
      if (c == row)
        continue;
      const int32_t q = inv[c];
      if ((q > place || (q == place && k > pos)) && q < best) {
        best = q;
        at = k;
      }
    }
    from = at;
    if (at < 0)
      return (I)0;
    place = best;
    pos = at;
    return (I)(best - i);
  };
  const int64_t at = (int64_t)poff[s] * 64 + lane;
  const int w = poff[s + 1] - poff[s];
  for (int q = 0; q < w; ++q) {
    int2 f;
    I2 d;
    d.x = next(f.x);
    d.y = next(f.y);
    reinterpret_cast<I2*>(idx)[at + (int64_t)q * 64] = d;
    reinterpret_cast<int2*>(src)[at + (int64_t)q * 64] = f;
  }
}

template <bool WANT32>
__global__ void __launch_bounds__(64)
k_pairp_values(int32_t n, const int32_t* __restrict__ perm, const int32_t* __restrict__ rp,
               const int32_t* __restrict__ ci, const double* __restrict__ v, const int32_t* __restrict__ poff,
               const int32_t* __restrict__ src, double* __restrict__ v64, double* __restrict__ diag64,
               double* __restrict__ dinv64, float* __restrict__ v32, float* __restrict__ diag32,
               float* __restrict__ dinv32)
{
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x;
  const int32_t i = s * 64 + lane;
  const int64_t at = (int64_t)poff[s] * 64 + lane;
  const int w = poff[s + 1] - poff[s];
  for (int q = 0; q < w; ++q) {
    const int2 f = reinterpret_cast<const int2*>(src)[at + (int64_t)q * 64];
    const double x = f.x >= 0 ? v[f.x] : 0.0, y = f.y >= 0 ? v[f.y] : 0.0;
    reinterpret_cast<double2*>(v64)[at + (int64_t)q * 64] = make_double2(x, y);
    if constexpr (WANT32)
      reinterpret_cast<float2*>(v32)[at + (int64_t)q * 64] = make_float2((float)x, (float)y);
  }
  if (i >= n)
    return;
  const int32_t row = perm[i];
  double diag = 0.0, sum = 0.0;
  for (int32_t k = rp[row]; k < rp[row + 1]; ++k) {
    sum += v[k];
    diag += ci[k] == row ? v[k] : 0.0;
  }
  const double inv = diag != 0.0 ? 1.0 / diag : 1.0;
  diag64[i] = diag;
  dinv64[i] = inv;
  if constexpr (WANT32) {
    diag32[i] = (float)sum;
    dinv32[i] = (float)inv;
  }
}

__device__ __forceinline__ uint32_t prec_bits(float f, bool bf16)
{
  const uint32_t u = __float_as_uint(f);
  if (!bf16)
    return u;
  return (u & 0x7fffffffu) > 0x7f800000u ? 0x7fc00000u : (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
}

template <bool BF16>
__global__ void __launch_bounds__(64)
k_pairp_prec(int32_t n, const int32_t* __restrict__ perm, const int32_t* __restrict__ rp,
             const int32_t* __restrict__ ci, const float* __restrict__ v, const int32_t* __restrict__ poff,
             const int32_t* __restrict__ src, uint32_t* __restrict__ out, float* __restrict__ mdiag)
{
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x;
  const int32_t i = s * 64 + lane;
  const int64_t at = (int64_t)poff[s] * 64 + lane;
  const int w = poff[s + 1] - poff[s];
  for (int q = 0; q < w; ++q) {
    const int2 f = reinterpret_cast<const int2*>(src)[at + (int64_t)q * 64];
    const uint32_t x = f.x >= 0 ? prec_bits(v[f.x], BF16) : 0u, y = f.y >= 0 ? prec_bits(v[f.y], BF16) : 0u;
    if constexpr (BF16)
      out[at + (int64_t)q * 64] = (x >> 16) | y;
    else
      reinterpret_cast<uint2*>(out)[at + (int64_t)q * 64] = make_uint2(x, y);
  }
  if (i >= n)
    return;
  const int32_t row = perm[i];
  float diag = 0.f;
  for (int32_t k = rp[row]; k < rp[row + 1]; ++k)
    diag += ci[k] == row ? __uint_as_float(prec_bits(v[k], BF16)) : 0.f;
  mdiag[i] = diag;
}

__global__ void k_permute_in(int32_t n, const int32_t* __restrict__ perm, const double* __restrict__ x,
                             const double* __restrict__ b, double* __restrict__ xp, double* __restrict__ bp)
{
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    xp[i] = x[perm[i]];
    bp[i] = b[perm[i]];
  }
}

__global__ void k_permute_out(int32_t n, const int32_t* __restrict__ perm, const double* __restrict__ xp,
                              double* __restrict__ x)
{
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    x[perm[i]] = xp[i];
}

// ---- offsets and values in the matrix's own order -----------------------------------------------

template <class I>
__global__ void __launch_bounds__(64)
k_pair_index(int32_t nslice, const int32_t* __restrict__ slice_row, const int32_t* __restrict__ rp,
             const int32_t* __restrict__ ci, const int32_t* __restrict__ poff, I* __restrict__ idx)
{
  typedef I I2 __attribute__((ext_vector_type(2)));
  __shared__ int32_t s_col[kStageMax];
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x;
  int32_t row, b, e, e0, e1;
  bool live;
  slice_rows(slice_row, nslice, s, rp, lane, row, live, b, e, e0, e1);
  const bool staged = e1 - e0 <= kStageMax;
  if (staged) {
    for (int32_t k = e0 + lane; k < e1; k += 64)
      s_col[k - e0] = ci[k];
    __syncthreads();
  }
  int32_t k = b;
  auto next = [&]() -> I { // offset of the row's next off-diagonal entry, 0 past the end
    while (k < e) {
      const int32_t c = staged ? s_col[k - e0] : ci[k];
      ++k;
      if (c != row)
        return (I)(c - row);
    }
    return (I)0;
  };
  I2* out = reinterpret_cast<I2*>(idx) + (int64_t)poff[s] * 64 + lane;
  const int w = poff[s + 1] - poff[s];
  for (int q = 0; q < w; ++q) {
    I2 d;
    d.x = next();
    d.y = next();
    out[(int64_t)q * 64] = d;
  }
}

// FP64 pairs, diagonal and its inverse, and (WANT32) the FP32 difference
// form: off-diagonal entries rounded, diag32 the row sum taken in FP64, so
// that y_i = diag32_i x_i + sum a_ij (x_j - x_i) has no rounded diagonal
// cancelling the other terms on smooth vectors.
template <bool WANT32>
__global__ void __launch_bounds__(64)
k_pair_values(int32_t nslice, const int32_t* __restrict__ slice_row, const int32_t* __restrict__ rp,
              const int32_t* __restrict__ ci, const double* __restrict__ v, const int32_t* __restrict__ poff,
              int stage, double* __restrict__ v64, double* __restrict__ diag64, double* __restrict__ dinv64,
              float* __restrict__ v32, float* __restrict__ diag32, float* __restrict__ dinv32)
{
  typedef double d2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  extern __shared__ __align__(16) unsigned char smem[]; // stage values, then stage columns
  double* s_val = reinterpret_cast<double*>(smem);
  int32_t* s_col = reinterpret_cast<int32_t*>(s_val + stage);
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x;
  int32_t row, b, e, e0, e1;
  bool live;
  slice_rows(slice_row, nslice, s, rp, lane, row, live, b, e, e0, e1);
  const bool staged = e1 - e0 <= stage;
  if (staged) {
    for (int32_t k = e0 + lane; k < e1; k += 64) {
      s_val[k - e0] = v[k];
      s_col[k - e0] = ci[k];
    }
    __syncthreads();
  }
  double diag = 0.0, sum = 0.0;
  int32_t k = b;
  auto next = [&]() -> double {
    while (k < e) {
      const int32_t c = staged ? s_col[k - e0] : ci[k];
      const double a = staged ? s_val[k - e0] : v[k];
      ++k;
      sum += a;
      if (c != row)
        return a;
      diag += a;
    }
    return 0.0;
  };
  const int64_t at = (int64_t)poff[s] * 64 + lane;
  const int w = poff[s + 1] - poff[s];
  for (int q = 0; q < w; ++q) {
    d2 m;
    m.x = next();
    m.y = next();
    reinterpret_cast<d2*>(v64)[at + (int64_t)q * 64] = m;
    if constexpr (WANT32)
      reinterpret_cast<f2*>(v32)[at + (int64_t)q * 64] = f2{ (float)m.x, (float)m.y };
  }
  (void)next(); // a diagonal entry after the last off-diagonal one
  if (live) {
    const double inv = diag != 0.0 ? 1.0 / diag : 1.0;
    diag64[row] = diag;
    dinv64[row] = inv;
    if constexpr (WANT32) {
      diag32[row] = (float)sum;
      dinv32[row] = (float)inv;
    }
  }
}

// Sparse preconditioner with the pattern of the matrix: FP32 pairs, or pairs
// of BF16 values (round to nearest even) in one word; its diagonal in FP32
// with the same rounding.
template <bool BF16>
__global__ void __launch_bounds__(64)
k_pair_prec(int32_t nslice, const int32_t* __restrict__ slice_row, const int32_t* __restrict__ rp,
            const int32_t* __restrict__ ci, const float* __restrict__ v, const int32_t* __restrict__ poff, int stage,
            uint32_t* __restrict__ out, float* __restrict__ mdiag)
{
  extern __shared__ __align__(16) unsigned char smem[]; // stage values, then stage columns
  float* s_val = reinterpret_cast<float*>(smem);
  int32_t* s_col = reinterpret_cast<int32_t*>(s_val + stage);
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x;
  int32_t row, b, e, e0, e1;
  bool live;
  slice_rows(slice_row, nslice, s, rp, lane, row, live, b, e, e0, e1);
  const bool staged = e1 - e0 <= stage;
  if (staged) {
    for (int32_t k = e0 + lane; k < e1; k += 64) {
      s_val[k - e0] = v[k];
      s_col[k - e0] = ci[k];
    }
    __syncthreads();
  }
  float diag = 0.f;
  int32_t k = b;
  auto next = [&]() -> uint32_t {
    while (k < e) {
      const int32_t c = staged ? s_col[k - e0] : ci[k];
      const uint32_t a = prec_bits(staged ? s_val[k - e0] : v[k], BF16);
      ++k;
      if (c != row)
        return a;
      diag += __uint_as_float(a);
    }
    return 0u;
  };
  const int64_t at = (int64_t)poff[s] * 64 + lane;
  const int w = poff[s + 1] - poff[s];
  for (int q = 0; q < w; ++q) {
    const uint32_t x = next(), y = next();
    if constexpr (BF16)
      out[at + (int64_t)q * 64] = (x >> 16) | y;
    else
      reinterpret_cast<uint2*>(out)[at + (int64_t)q * 64] = make_uint2(x, y);
  }
  (void)next(); // a diagonal entry after the last off-diagonal one
  if (live)
    mdiag[row] = diag;
}

// ---- launch layout ------------------------------------------------------------------------------

// A workgroup takes a slice for each of its waves before a team gets another:
// 66 thousand rows on 65 workgroups 6.3 us an iteration, on 130 7.1, on 256 8.0
// (the barriers).
static int waves_of(const Pack& p) { return p.block == 3 ? kBlockWaves : kWaves; }
static int max_rows(const Pack& p) { return p.block == 3 ? kBlockRowSteps[2] : kRowSteps[3]; }
// Iterations of one launch: 0.05 s for a system of 66 thousand rows, 0.3 s for
// 2.15 million of tetrahedra, 4 s for the largest layout that is accepted (2.5
// GiB of FP64 pairs and offsets an iteration).
constexpr int kLaunchIterations = 8192;

// Workgroups a segment needs at least (max_rows slices per wave).
static int32_t least_workgroups(const Pack& p, int k)
{
  const int32_t sl = p.seg_slices[k + 1] - p.seg_slices[k];
  const int32_t most = waves_of(p) * max_rows(p);
  return (sl + most - 1) / most;
}

// Workgroups per segment of `segs`, `budget` together: at least what it needs,
// at most one slice per wave, else in proportion to rows^1.5 (the work of an
// iteration times the growth of the iteration count).
static std::vector<int32_t> team_sizes(const Pack& p, const std::vector<int>& segs, int budget)
{
  const size_t ns = segs.size();
  const int waves = waves_of(p);
  std::vector<int32_t> m(ns);
  std::vector<double> w(ns);
  double wsum = 0.0;
  for (size_t i = 0; i < ns; ++i) {
    w[i] = std::pow((double)(p.seg_rows[segs[i] + 1] - p.seg_rows[segs[i]]), 1.5);
    wsum += w[i];
  }
  for (double scale = budget;; scale *= 0.97) {
    int64_t total = 0;
    for (size_t i = 0; i < ns; ++i) {
      const int32_t sl = p.seg_slices[segs[i] + 1] - p.seg_slices[segs[i]];
      m[i] = std::max(least_workgroups(p, segs[i]),
                      std::min<int32_t>((sl + waves - 1) / waves, (int32_t)std::floor(scale * w[i] / wsum)));
      total += m[i];
    }
    if (total <= budget)
      return m;
  }
}

static size_t diagonal_values(const Pack& p)
{
  return p.block == 3 ? (size_t)p.nslice * 64 * 9 : (size_t)p.n;
}

// ---- building the pair layout -------------------------------------------------------------------

bool pack_pattern(Pack& p, int32_t n, int64_t nnz, const int32_t* rp, const int32_t* ci,
                  const std::vector<int32_t>& seg_rows, const int32_t* order, int block)
{
  p.n = n;
  p.block = block;
  p.valid64 = p.valid32 = false;
  p.valid_prec = 0;
  p.seg_rows = seg_rows;
  const int nseg = (int)seg_rows.size() - 1;
  p.seg_slices.assign(nseg + 1, 0);
  for (int k = 0; k < nseg; ++k)
    p.seg_slices[k + 1] = p.seg_slices[k] + (seg_rows[k + 1] - seg_rows[k] + 63) / 64;
  p.nslice = p.seg_slices[nseg];
  for (int k = 0; k < nseg; ++k)
    if (least_workgroups(p, k) > rt().num_cu)
      return false;
  std::vector<int32_t> sr((size_t)3 * p.nslice);
  for (int k = 0; k < nseg; ++k)
    for (int32_t s = p.seg_slices[k]; s < p.seg_slices[k + 1]; ++s) {
      sr[s] = seg_rows[k] + 64 * (s - p.seg_slices[k]);
      sr[(size_t)p.nslice + s] = seg_rows[k];
      sr[(size_t)2 * p.nslice + s] = seg_rows[k + 1];
    }
  p.slice_row.reserve(sr.size());
  p.slice_row.upload(sr.data(), sr.size());
  DBuf<int32_t> width((size_t)p.nslice), stats(4);
  stats.zero();
  hipLaunchKernelGGL(k_pair_count, dim3(p.nslice), dim3(64), 0, stream(), p.nslice, p.slice_row.p, rp, ci, width.p,
                     stats.p);
  check_launch("pair_count");
  int32_t h[4];
  stats.download(h, 4);
  // Numbered at random (as a mesh generator's nodes come), a gather of 64 rows
  // touches about 60 lines of the published vector; in Morton order of the
  // nodes about 14, numbered along a grid 6 (tetrahedra, FP64, 118 thousand
  // rows: 16.6 -> 9.9 us an iteration).  Numbered along a grid, the matrix
  // keeps its order: Morton order would read more lines.
  p.perm.release();
  if (order && nseg == 1 && block == 1 && 2 * h[3] > p.nslice) {
    p.perm.alloc((size_t)n);
    p.inv.reserve((size_t)n);
    AFEM_HIP(hipMemcpyAsync(p.perm.p, order, sizeof(int32_t) * (size_t)n, hipMemcpyDeviceToDevice, stream()));
    hipLaunchKernelGGL(k_invert, dim3(grid_for(n, 256)), dim3(256), 0, stream(), n, p.perm.p, p.inv.p);
    stats.zero();
    hipLaunchKernelGGL(k_pairp_count, dim3(p.nslice), dim3(64), 0, stream(), p.nslice, n, p.perm.p, p.inv.p, rp, ci,
                       width.p, stats.p);
    check_launch("pairp_count");
    int32_t far[2];
    stats.download(far, 2);
    h[1] = far[1];
  }
  p.poff.reserve((size_t)p.nslice + 1);
  p.npair = exclusive_scan_i32(width.p, p.poff.p, p.nslice);
  // a segment's buffers end with its rows; a few long rows would pad their slices many times over, and the kernel's
  // stream offsets are 31 bits wide
  if ((h[2] & 2) || p.npair * 128 > 4 * nnz + 65536 || p.npair * (kWave * 16) * (block * block) >= (1LL << 31))
    return false;
  p.max_len = h[0];
  p.idx16 = h[1] <= 32767;
  p.all_diag = (h[2] & 1) == 0;
  p.idx.reserve((size_t)p.npair * (p.idx16 ? 64 : 128));
  p.v64.reserve((size_t)p.npair * 128 * (block * block));
  p.diag64.reserve(diagonal_values(p));
  p.dinv64.reserve(diagonal_values(p));
  if (p.perm.p) {
    p.src.reserve((size_t)p.npair * 128);
    if (p.idx16)
      hipLaunchKernelGGL(k_pairp_index<int16_t>, dim3(p.nslice), dim3(64), 0, stream(), n, p.perm.p, p.inv.p, rp, ci,
                         p.poff.p, reinterpret_cast<int16_t*>(p.idx.p), p.src.p);
    else
      hipLaunchKernelGGL(k_pairp_index<int32_t>, dim3(p.nslice), dim3(64), 0, stream(), n, p.perm.p, p.inv.p, rp, ci,
                         p.poff.p, p.idx.p, p.src.p);
    check_launch("pairp_index");
  }
  else if (p.npair > 0) {
    if (p.idx16)
      hipLaunchKernelGGL(k_pair_index<int16_t>, dim3(p.nslice), dim3(64), 0, stream(), p.nslice, p.slice_row.p, rp,
                         ci, p.poff.p, reinterpret_cast<int16_t*>(p.idx.p));
    else
      hipLaunchKernelGGL(k_pair_index<int32_t>, dim3(p.nslice), dim3(64), 0, stream(), p.nslice, p.slice_row.p, rp,
                         ci, p.poff.p, p.idx.p);
    check_launch("pair_index");
  }
  return true;
}

void pack_values(Pack& p, const int32_t* rp, const int32_t* ci, const double* v, bool want32)
{
  if (p.valid64 && (p.valid32 || !want32))
    return;
  if (want32) {
    p.v32.reserve((size_t)p.npair * 128 * (p.block * p.block));
    p.diag32.reserve(diagonal_values(p));
    p.dinv32.reserve(diagonal_values(p));
  }
  const int stage = std::min(kStageMax, std::max(1, p.max_len) * 64);
  const size_t lds = (size_t)stage * 12;
  if (p.block == 3)
    fill_block_values(p, rp, ci, v, want32);
  else if (p.perm.p && want32)
    hipLaunchKernelGGL(k_pairp_values<true>, dim3(p.nslice), dim3(64), 0, stream(), p.n, p.perm.p, rp, ci, v, p.poff.p,
                       p.src.p, p.v64.p, p.diag64.p, p.dinv64.p, p.v32.p, p.diag32.p, p.dinv32.p);
  else if (p.perm.p)
    hipLaunchKernelGGL(k_pairp_values<false>, dim3(p.nslice), dim3(64), 0, stream(), p.n, p.perm.p, rp, ci, v,
                       p.poff.p, p.src.p, p.v64.p, p.diag64.p, p.dinv64.p, (float*)nullptr, (float*)nullptr,
                       (float*)nullptr);
  else if (want32)
    hipLaunchKernelGGL(k_pair_values<true>, dim3(p.nslice), dim3(64), lds, stream(), p.nslice, p.slice_row.p, rp, ci,
                       v, p.poff.p, stage, p.v64.p, p.diag64.p, p.dinv64.p, p.v32.p, p.diag32.p, p.dinv32.p);
  else
    hipLaunchKernelGGL(k_pair_values<false>, dim3(p.nslice), dim3(64), lds, stream(), p.nslice, p.slice_row.p, rp, ci,
                       v, p.poff.p, stage, p.v64.p, p.diag64.p, p.dinv64.p, (float*)nullptr, (float*)nullptr,
                       (float*)nullptr);
  check_launch("pair_values");
  p.valid64 = true;
  p.valid32 = p.valid32 || want32;
}

void reserve(Work& w, int nseg)
{
  if (w.nseg >= nseg && w.host)
    return;
  if (w.host)
    AFEM_HIP(hipHostFree(w.host));
  w.host = nullptr;
  AFEM_HIP(hipHostMalloc(reinterpret_cast<void**>(&w.host), sizeof(Status) * ((size_t)nseg + 1),
                         hipHostMallocDefault));
  w.st.alloc((size_t)nseg + 1);
  w.nseg = nseg;
}

__global__ void k_clear_slots(int64_t n, uint64_t* __restrict__ slots)
{
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    slots[i] = 0;
}

// Rounds of segments, the largest first: a round takes segments while the
// workgroups that they need at least fit the device together.
static std::vector<std::vector<int>> rounds_of(const Pack& p, int budget)
{
  const int ns = (int)p.seg_rows.size() - 1;
  std::vector<int> order(ns);
  for (int k = 0; k < ns; ++k)
    order[k] = k;
  std::stable_sort(order.begin(), order.end(), [&](int i, int j) {
    return p.seg_rows[i + 1] - p.seg_rows[i] > p.seg_rows[j + 1] - p.seg_rows[j];
  });
  std::vector<std::vector<int>> out;
  int need = budget + 1;
  for (int k : order) {
    const int m = least_workgroups(p, k);
    if (need + m > budget) {
      out.emplace_back();
      need = 0;
    }
    out.back().push_back(k);
    need += m;
  }
  return out;
}

int round_count(const Pack& p) { return (int)rounds_of(p, rt().num_cu).size(); }

static void layout(const Pack& p, Work& w)
{
  if (!w.rounds.empty() && w.layout_rows == p.seg_rows)
    return;
  const int budget = rt().num_cu;
  constexpr int kTeamWords = sizeof(TeamDesc) / sizeof(int32_t);
  std::vector<int32_t> out;
  w.rounds.clear();
  int64_t slot = 0;
  for (const std::vector<int>& segs : rounds_of(p, budget)) {
    const std::vector<int32_t> m = team_sizes(p, segs, budget);
    Round r;
    r.first_word = (int)out.size();
    r.teams = (int)segs.size();
    r.first_slot = slot;
    int rows = 1;
    for (size_t i = 0; i < segs.size(); ++i) {
      const int k = segs[i];
      const int32_t sl = p.seg_slices[k + 1] - p.seg_slices[k];
      const TeamDesc t{ p.seg_rows[k], p.seg_rows[k + 1], p.seg_slices[k], sl, r.grid, m[i], k, 0 };
      const int32_t* q = reinterpret_cast<const int32_t*>(&t);
      out.insert(out.end(), q, q + kTeamWords);
      const int per_wg = (sl + m[i] - 1) / m[i];
      rows = std::max(rows, (per_wg + waves_of(p) - 1) / waves_of(p));
      r.grid += m[i];
    }
    for (size_t i = 0; i < segs.size(); ++i)
      out.insert(out.end(), (size_t)m[i], (int32_t)i);
    out.resize((out.size() + kTeamWords - 1) / kTeamWords * kTeamWords);
    const auto at_least = [&](int q) { return q >= rows; };
    r.rows_per_wave = p.block == 3
      ? *std::find_if(std::begin(kBlockRowSteps), std::end(kBlockRowSteps), at_least)
      : *std::find_if(std::begin(kRowSteps), std::end(kRowSteps), at_least);
    slot += (int64_t)2 * r.grid * kSlotWords;
    w.rounds.push_back(r);
  }
  w.team.reserve(out.size());
  w.team.upload(out.data(), out.size());
  w.slots.release();
  w.layout_rows = p.seg_rows;
}

bool solve(const Pack& p, Work& w, const Options& o, double* x, const double* b)
{
  const int ns = (int)p.seg_rows.size() - 1;
  layout(p, w);
  const size_t dofs = (size_t)p.n * p.block;
  w.u.reserve(dofs);
  w.keep.reserve(3 * dofs);
  if (!w.slots.p || w.epoch > 0x40000000u) {
    w.slots.reserve((size_t)(w.rounds.back().first_slot + (int64_t)2 * w.rounds.back().grid * kSlotWords));
    hipLaunchKernelGGL(k_clear_slots, dim3(64), dim3(256), 0, stream(), (int64_t)w.slots.n, w.slots.p);
    check_launch("resident_clear");
    w.epoch = 0;
  }
  Args a{};
  a.poff = p.poff.p;
  a.idx = p.idx.p;
  a.v = o.mixed ? (const void*)p.v32.p : (const void*)p.v64.p;
  a.diag = o.mixed ? (const void*)p.diag32.p : (const void*)p.diag64.p;
  a.dinv = o.mixed ? (const void*)p.dinv32.p : (const void*)p.dinv64.p;
  a.m = p.m.p;
  a.mdiag = p.mdiag.p;
  a.v64 = p.v64.p;
  a.diag64 = p.diag64.p;
  a.x = x;
  a.b = b;
  if (p.perm.p) {
    w.xb.reserve(2 * dofs);
    a.x = w.xb.p;
    a.b = w.xb.p + dofs;
    ProfScope prof("resident_reorder");
    hipLaunchKernelGGL(k_permute_in, dim3(grid_for(p.n, 256)), dim3(256), 0, stream(), p.n, p.perm.p, x, b, w.xb.p,
                       w.xb.p + dofs);
    check_launch("permute_in");
  }
  a.u = w.u.p;
  a.keep = w.keep.p;
  a.n = p.n;
  a.st = w.st.p;
  a.abort_flag = &w.st.p[ns].done;
  a.spin_limit = o.spin_limit > 0 ? o.spin_limit : (1LL << 22);
  a.precond = o.precond ? 1 : 0;
  a.norm = o.norm;
  a.max_launch_iter = kLaunchIterations;
  for (int k = 0; k < ns; ++k) {
    Status& s = w.host[k];
    s.iter = s.done = s.converged = s.breakdown = s.nb_ru = 0;
    s.bb = s.rr_out = s.rr_true = s.rho = s.rr_ref = s.beta = 0.0;
  }
  for (;;) {
    w.host[ns] = Status{};
    for (int k = 0; k < ns; ++k)
      w.host[k].epoch = w.epoch;
    AFEM_HIP(hipMemcpyAsync(w.st.p, w.host, sizeof(Status) * ((size_t)ns + 1), hipMemcpyHostToDevice, stream()));
    for (const Round& r : w.rounds) {
      a.team = reinterpret_cast<const TeamDesc*>(w.team.p + r.first_word);
      a.team_of = w.team.p + r.first_word + (size_t)r.teams * (sizeof(TeamDesc) / sizeof(int32_t));
      a.slots = w.slots.p + r.first_slot;
      const size_t lds = (size_t)r.rows_per_wave * kBS * 16; // x, and D^-1 (FP64) or p (mixed)
      ProfScope prof(o.prec ? "resident_fpcg" : o.mixed ? "resident_cg_mixed" : "resident_cg_fp64");
      if (p.block == 3)
        launch_block(a, o.mixed, r.rows_per_wave, p.idx16, r.grid);
      else if (o.prec)
        launch_flex(a, r.rows_per_wave, p.idx16, o.prec == 16, r.grid, lds);
      else if (o.mixed)
        launch_f32(a, r.rows_per_wave, p.idx16, r.grid, lds);
      else
        launch_f64(a, r.rows_per_wave, p.idx16, r.grid, lds);
    }
    if (p.perm.p) {
      hipLaunchKernelGGL(k_permute_out, dim3(grid_for(p.n, 256)), dim3(256), 0, stream(), p.n, p.perm.p, a.x, x);
      check_launch("permute_out");
    }
    AFEM_HIP(hipMemcpyAsync(w.host, w.st.p, sizeof(Status) * ((size_t)ns + 1), hipMemcpyDeviceToHost, stream()));
    AFEM_HIP(hipStreamSynchronize(stream()));
    if (w.host[ns].done) { // a wait gave up: slots of unknown epochs
      w.slots.release();
      return false;
    }
    bool all = true;
    for (int k = 0; k < ns; ++k) {
      w.epoch = std::max(w.epoch, w.host[k].epoch);
      all = all && (!w.host[k].active || w.host[k].done);
    }
    if (all)
      return true;
    a.resume = 1;
  }
}

void pack_prec(Pack& p, const int32_t* rp, const int32_t* ci, const float* v, int bits)
{
  if (p.valid_prec == bits)
    return;
  p.m.reserve((size_t)p.npair * (bits == 16 ? 64 : 128));
  p.mdiag.reserve((size_t)p.n);
  const int stage = std::min(kStageMax, std::max(1, p.max_len) * 64);
  const size_t lds = (size_t)stage * 8;
  if (p.perm.p && bits == 16)
    hipLaunchKernelGGL(k_pairp_prec<true>, dim3(p.nslice), dim3(64), 0, stream(), p.n, p.perm.p, rp, ci, v, p.poff.p,
                       p.src.p, p.m.p, p.mdiag.p);
  else if (p.perm.p)
    hipLaunchKernelGGL(k_pairp_prec<false>, dim3(p.nslice), dim3(64), 0, stream(), p.n, p.perm.p, rp, ci, v, p.poff.p,
                       p.src.p, p.m.p, p.mdiag.p);
  else if (bits == 16)
    hipLaunchKernelGGL(k_pair_prec<true>, dim3(p.nslice), dim3(64), lds, stream(), p.nslice, p.slice_row.p, rp, ci, v,
                       p.poff.p, stage, p.m.p, p.mdiag.p);
  else
    hipLaunchKernelGGL(k_pair_prec<false>, dim3(p.nslice), dim3(64), lds, stream(), p.nslice, p.slice_row.p, rp, ci,
                       v, p.poff.p, stage, p.m.p, p.mdiag.p);
  check_launch("pair_prec");
  p.valid_prec = bits;
}

void launch_f64(const Args& a, int rows, bool idx16, int grid, size_t lds)
{
  if (idx16)
    launch_kernel<double, 0, true>(a, rows, grid, lds);
  else
    launch_kernel<double, 0, false>(a, rows, grid, lds);
}

} // namespace resident
} // namespace afem
