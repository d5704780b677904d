// resident_kernel.h -- the resident conjugate-gradient kernel (see resident.hip).
#pragma once

#include "device_utils.h"
#include "resident.h"

namespace afem {
namespace resident {

// One workgroup per CU, 1024 threads of 128 registers: against 512 threads of
// 256 registers twice the waves hide the gathers' latency (24 systems of
// triangles 12.9 -> 10.3 us an iteration, 227 thousand rows of tetrahedra
// FP64 13.4 -> 11.6, 2.15 million rows mixed 42.8 -> 40.4, with the mixed
// solver's terms still rounded to FP32), at the price of
// some spills at 9 slices per wave.
constexpr int kBS = 1024;
constexpr int kWaves = kBS / kWave;
constexpr int kSlotWords = 8; // 64 bytes per workgroup and parity

struct TeamDesc // the workgroups of one segment
{
  int32_t row0, row1, slice0, nslice, wg0, nwg, seg, pad;
};

struct Args
{
  const TeamDesc* team;
  const int32_t* team_of; // team of each workgroup
  const int32_t* poff;
  const int32_t* idx;
  const void* v;    // pairs of the product: FP64, or FP32 in difference form
  const void* diag; // its diagonal
  const void* dinv;
  const void* m;     // pairs of the sparse preconditioner (FP32 or BF16) and its diagonal
  const float* mdiag;
  const double* v64; // FP64 pairs and diagonal of the residual
  const double* diag64;
  double* x;
  const double* b;
  void* u;      // published u = D r, or z then r with a sparse preconditioner
  double* keep; // r, p, s (n each)
  int32_t n;
  uint64_t* slots;
  int32_t* abort_flag;
  Status* st;
  long long spin_limit;
  int precond, norm, resume, max_launch_iter;
};

typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// ---- exchange through the device's coherence point ------------------------------------------
//
// The published vector is written and read with agent-scope accesses (the sc1
// bit of buffer loads and stores), so no cache is written back or invalidated
// at a barrier and the matrix stays in the L2.  Buffers cover the rows of one
// segment: a lane past its end reads zeros and writes nothing, so partial
// slices need no masks.

constexpr int kSc1 = 16;
using Rsrc = __amdgpu_buffer_rsrc_t;

template <class T>
__device__ __forceinline__ Rsrc segment_buffer(const T* p, int32_t row0, int32_t rows)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p) + row0, 0, (int)((uint32_t)rows * (uint32_t)sizeof(T)),
                                           0x00027000);
}

// AUX: 0 ordinary cached access, kSc1 through the coherence point.  `row` is
// relative to the segment.
template <class T, int AUX>
__device__ __forceinline__ T bload(Rsrc r, int32_t row)
{
  // the whole offset in one register: no part of it moves to the immediate
  // field, where a negative rest would be out of range
  uint32_t off = (uint32_t)row * (uint32_t)sizeof(T);
  asm("" : "+v"(off));
  if constexpr (sizeof(T) == 4)
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, AUX));
  else {
    const v2u w = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, AUX);
    return __longlong_as_double((long long)(((uint64_t)w.y << 32) | w.x));
  }
}

template <class T, int AUX>
__device__ __forceinline__ void bstore(Rsrc r, int32_t row, T v)
{
  const uint32_t off = (uint32_t)row * (uint32_t)sizeof(T);
  if constexpr (sizeof(T) == 4)
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)off, 0, AUX);
  else {
    const uint64_t q = (uint64_t)__double_as_longlong(v);
    __builtin_amdgcn_raw_buffer_store_b64(v2u{ (uint32_t)q, (uint32_t)(q >> 32) }, r, (int)off, 0, AUX);
  }
}

// ---- sums ---------------------------------------------------------------------------------------

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v)
{
  const uint64_t q = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)q, CTRL, ROWS, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(q >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Sum over the wave, in lane 63: shifts within rows of 16 lanes, then the
// rows' last lanes broadcast on (register moves, no LDS round trips).
__device__ __forceinline__ double wave_sum63(double v)
{
  v = dpp_add<0x111, 0xf>(v); // row_shr:1
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v); // row_bcast:15
  v = dpp_add<0x143, 0xc>(v); // row_bcast:31
  return v;
}

__device__ __forceinline__ double lane63(double v)
{
  const uint64_t q = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)q, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(q >> 32), 63);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

struct Barrier
{
  uint64_t* base;  // this team's slots, parity 0
  int64_t parity;  // words between the parities
  int32_t* abort_flag;
  long long limit;
  int me, nwg;
  unsigned epoch;
};

// Team-wide barrier that sums NV numbers over the team.  A workgroup writes
// its sums into its slot as words {epoch << 32 | half of a double}; a word of
// the current epoch is valid by itself, so one store and one poll replace the
// arrival counter, its polling and the reading of the partial sums.  Slots
// alternate between two sets: a set is written again only after every
// workgroup has passed the barrier after it.  All workgroups add the slots in
// the same order and hold the same sums.  False: a wait gave up.
template <int NV, int WAVES = kWaves>
__device__ __forceinline__ bool team_sum(Barrier& B, double (&v)[NV])
{
  static_assert(2 * NV <= kSlotWords, "slot too small");
  __shared__ double s_part[NV][WAVES];
  __shared__ double s_tot[NV];
  __shared__ int s_ok;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const unsigned epoch = ++B.epoch;
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const double s = wave_sum63(v[q]);
    if (lane == kWave - 1)
      s_part[q][wave] = s;
  }
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0); // this wave's published values are acknowledged
  __syncthreads();
  if (wave == 0) {
    uint64_t* base = B.base + (epoch & 1) * B.parity;
    if (lane < 2 * NV) {
      const int q = lane >> 1;
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w)
        s += s_part[q][w];
      const uint64_t u = (uint64_t)__double_as_longlong(s);
      const uint32_t half = (lane & 1) ? (uint32_t)(u >> 32) : (uint32_t)u;
      __hip_atomic_store(base + (int64_t)B.me * kSlotWords + lane, ((uint64_t)epoch << 32) | half, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
    double acc[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q)
      acc[q] = 0.0;
    int ok = 1;
    for (int g = lane; g < B.nwg; g += kWave) {
      const uint64_t* s = base + (int64_t)g * kSlotWords;
      uint64_t w[2 * NV];
      long long polls = 0;
      for (;;) {
        bool all = true;
#pragma unroll
        for (int q = 0; q < 2 * NV; ++q)
          w[q] = __hip_atomic_load(const_cast<uint64_t*>(s) + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int q = 0; q < 2 * NV; ++q)
          all = all && (uint32_t)(w[q] >> 32) == epoch;
        if (all)
          break;
        ++polls;
        if (polls >= B.limit ||
            ((polls & 1023) == 0 &&
             __hip_atomic_load(B.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          ok = 0;
          break;
        }
      }
      if (!ok) {
        __hip_atomic_fetch_max(B.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
#pragma unroll
      for (int q = 0; q < NV; ++q)
        acc[q] += __longlong_as_double((long long)((w[2 * q] & 0xffffffffull) | (w[2 * q + 1] << 32)));
    }
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const double t = wave_sum63(acc[q]);
      if (lane == kWave - 1)
        s_tot[q] = t;
    }
    if (__all(ok) && lane == 0)
      s_ok = 1;
    else if (!__all(ok) && lane == 0)
      s_ok = 0;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q)
    v[q] = s_tot[q];
  return s_ok != 0;
}

// ---- matrix pairs -----------------------------------------------------------------------------------

// Two values and two offsets of a lane, read by one load each: the buffer's
// base and the pair number are scalars, so a stream costs no address registers.
template <class T>
struct ValuePair
{
  T x, y;
};

__device__ __forceinline__ Rsrc whole_buffer(const void* p)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, -1, 0x00027000);
}

template <class T>
__device__ __forceinline__ ValuePair<T> load_values(Rsrc r, int lane, int q)
{
  if constexpr (sizeof(T) == 4) {
    const v2u w = __builtin_amdgcn_raw_buffer_load_b64(r, lane * 8, q * (kWave * 8), 0);
    return { __uint_as_float(w.x), __uint_as_float(w.y) };
  }
  else {
    const v4u w = __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, q * (kWave * 16), 0);
    return { __longlong_as_double((long long)(((uint64_t)w.y << 32) | w.x)),
             __longlong_as_double((long long)(((uint64_t)w.w << 32) | w.z)) };
  }
}

template <bool I16>
struct IndexPair;
template <>
struct IndexPair<true>
{
  uint32_t w;
  __device__ __forceinline__ int x() const { return (int)(int16_t)(w & 0xffffu); }
  __device__ __forceinline__ int y() const { return (int)w >> 16; }
};
template <>
struct IndexPair<false>
{
  v2u w;
  __device__ __forceinline__ int x() const { return (int)w.x; }
  __device__ __forceinline__ int y() const { return (int)w.y; }
};

template <bool I16>
__device__ __forceinline__ IndexPair<I16> load_offsets(Rsrc r, int lane, int q)
{
  if constexpr (I16)
    return { __builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, q * (kWave * 4), 0) };
  else
    return { __builtin_amdgcn_raw_buffer_load_b64(r, lane * 8, q * (kWave * 8), 0) };
}

// ---- the kernel -------------------------------------------------------------------------------------

// One launch of preconditioned conjugate gradients.  Every wave owns up to R
// consecutive slices of its segment; each lane one row per slice.
//
//   A  w = A u; p = u + beta p; s = w + beta s (= A p); partial p.s
//   -- sum --
//   B  alpha = rho / p.s; x += alpha p; r -= alpha s; u = D r, published;
//      partials r.u, r.r
//   -- sum --   beta = r.u / rho; convergence
//
// With s kept by its recurrence the product reads u, which was published
// before the sum that gives beta, so an iteration has two barriers.  The mixed
// solver (T = float) has u and the matrix in FP32 and takes reliable updates:
// x is published, r = b - A64 x formed, u = D r published again.  Its r, p and
// s are FP64 and the terms of w exact (FP64 products of the FP32 numbers,
// summed in FP64): w is a product with the rough u, not with the smooth p, and
// what it loses stays in s.  With r and the products in FP32 the residual of a
// late reliable update differed from the recursive one by up to 0.4 %, which
// cost iterations and left more error at the same residual: checkerboard of
// 509 x 509 quads 4994 iterations, now 3320 (FP64 r alone: 4954); log-normal
// cube of 128^3 hexes 1572 (x error 1e-9; FP64 r alone 1724), now 1449 (6e-12;
// FP64 PCG takes 1448).  The price at 9 slices per wave is 40.8 -> 41.2 us an
// iteration at 2.15 million rows; at 5 there is none (16.8, 16.5 at 0.53
// million).
//
// With a sparse preconditioner (PREC 32 or 16: its values FP32 or BF16) B
// publishes r, and a third phase forms u = M r, published, and the partials
// u.r and u.s, whose sum gives the flexible beta = -alpha u.s / rho
// (Polak-Ribiere; u.r / rho after a reliable update).
//
// r, s, FP64's p and FP32's D^-1 (or u = M r) are in registers, and the
// diagonal but for the mixed solvers at 9 slices, which read it with the row's
// matrix (loaded after the row's sums instead: 42.1 us).  x, FP32's p and
// FP64's D^-1 are in LDS.  The matrices are the only other streams of an
// iteration: read a chunk of CP pairs ahead of their use, the first chunk of
// the next product ahead of the barriers.
enum StreamKind
{
  kStreamA = 0,
  kStreamM32 = 32,
  kStreamM16 = 16
};

template <class T, int R, bool I16, int PREC>
__global__ void __launch_bounds__(kBS, 4) k_cg(Args a)
{
  using V2 = ValuePair<T>;
  using I2 = IndexPair<I16>;
  constexpr bool MIXED = sizeof(T) == 4;
  constexpr bool FLEX = PREC != 0;
  static_assert(!FLEX || MIXED, "the sparse preconditioner is FP32");
  constexpr bool DLDS = !MIXED; // D^-1 in LDS and p in registers, else the other way round
  constexpr bool GREG = !MIXED || R <= 5; // the diagonal in registers
  constexpr int CP = MIXED ? 4 : (R > 5 ? 2 : 4);
  extern __shared__ __align__(16) unsigned char smem[];

  const int wg = (int)xcd_tile(blockIdx.x, gridDim.x);
  const TeamDesc team = a.team[a.team_of[wg]];
  Status& st = a.st[team.seg];
  if (!st.active || st.done)
    return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int me = wg - team.wg0;

  // this wave's slices
  const int64_t g0 = (int64_t)team.nslice * me / team.nwg, g1 = (int64_t)team.nslice * (me + 1) / team.nwg;
  const int s0 = (int)(g0 + (g1 - g0) * wave / kWaves);
  const int nsl = (int)(g0 + (g1 - g0) * (wave + 1) / kWaves) - s0;
  const int32_t row_first = s0 * kWave + lane; // within the segment, as every row below
  // slice offsets of the wave in the lanes of one register
  const int32_t po = a.poff[team.slice0 + s0 + min(lane, nsl)];
  auto pair0 = [&](int j) { return __builtin_amdgcn_readlane(po, j); };
  auto row_of = [&](int j) { return row_first + j * kWave; };

  Barrier bar;
  bar.base = a.slots + (int64_t)team.wg0 * kSlotWords;
  bar.parity = (int64_t)gridDim.x * kSlotWords;
  bar.abort_flag = a.abort_flag;
  bar.limit = a.spin_limit;
  bar.me = me;
  bar.nwg = team.nwg;
  bar.epoch = st.epoch;

  const int32_t rows = team.row1 - team.row0;
  const Rsrc urs = segment_buffer(reinterpret_cast<const T*>(a.u), team.row0, rows);
  const Rsrc rrs = segment_buffer(reinterpret_cast<const T*>(a.u) + (FLEX ? a.n : 0), team.row0, rows);
  const Rsrc xrs = segment_buffer(a.x, team.row0, rows);
  const Rsrc brs = segment_buffer(a.b, team.row0, rows);
  const Rsrc vrs = whole_buffer(a.v), irs = whole_buffer(a.idx), mrs = whole_buffer(a.m);
  const Rsrc mds = segment_buffer(a.mdiag, team.row0, FLEX ? rows : 0);

  double* l_x = reinterpret_cast<double*>(smem) + threadIdx.x;
  double* l_2 = l_x + R * kBS;
  T dg[GREG ? R : 1], di[DLDS ? 1 : R]; // FLEX: di holds u
  double r[R], s[R], pr[DLDS ? R : 1];
  auto get_p = [&](int j) -> double {
    if constexpr (DLDS)
      return pr[j];
    else
      return l_2[j * kBS];
  };
  auto set_p = [&](int j, double v) {
    if constexpr (DLDS)
      pr[j] = v;
    else
      l_2[j * kBS] = v;
  };
  auto get_d = [&](int j) -> T {
    if constexpr (DLDS)
      return l_2[j * kBS];
    else
      return di[j];
  };
  auto get_u = [&](int j) -> T { return FLEX ? di[DLDS ? 0 : j] : get_d(j) * (T)r[j]; };
  const Rsrc grs = segment_buffer(reinterpret_cast<const T*>(a.diag), team.row0, rows);
  auto get_g = [&](int j) -> T { return GREG ? dg[GREG ? j : 0] : bload<T, 0>(grs, row_of(j)); };
  {
    const Rsrc drs = segment_buffer(reinterpret_cast<const T*>(a.dinv), team.row0, rows);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      r[j] = s[j] = 0.0;
      if constexpr (GREG)
        dg[j] = (T)0;
      set_p(j, 0.0);
      if constexpr (!DLDS)
        di[j] = (T)0;
      if (j < nsl) {
        l_x[j * kBS] = bload<double, 0>(xrs, row_of(j));
        if constexpr (!FLEX) {
          const T d = a.precond ? bload<T, 0>(drs, row_of(j)) : (T)1;
          if constexpr (DLDS)
            l_2[j * kBS] = d;
          else
            di[j] = d;
        }
        if constexpr (GREG)
          dg[j] = bload<T, 0>(grs, row_of(j));
      }
    }
  }

  // b - A64 x of row j, x as published; 0 in the lanes past the segment
  auto residual = [&](int j) -> double {
    const Rsrc mrs64 = whole_buffer(a.v64);
    const Rsrc grs64 = segment_buffer(a.diag64, team.row0, rows);
    const int32_t row = row_of(j);
    double t0 = bload<double, 0>(grs64, row) * l_x[j * kBS], t1 = 0.0;
    const int q1 = pair0(j + 1);
    for (int q = pair0(j); q < q1; ++q) {
      const ValuePair<double> m = load_values<double>(mrs64, lane, q);
      const I2 d = load_offsets<I16>(irs, lane, q);
      t0 += m.x * bload<double, kSc1>(xrs, row + d.x());
      t1 += m.y * bload<double, kSc1>(xrs, row + d.y());
    }
    return bload<double, 0>(brs, row) - (t0 + t1);
  };
  auto publish_x = [&]() {
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl)
        bstore<double, kSc1>(xrs, row_of(j), l_x[j * kBS]);
  };

  // the stream: the chunk whose gathers go out next
  V2 cv[CP];
  I2 cd[CP];
  auto fetch = [&](auto stream, int q0, int cnt) {
    constexpr int S = decltype(stream)::value;
#pragma unroll
    for (int z = 0; z < CP; ++z)
      if (z < cnt) {
        if constexpr (S == kStreamM16)
          cv[z].x = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(mrs, lane * 4, (q0 + z) * (kWave * 4), 0));
        else
          cv[z] = load_values<T>(S == kStreamA ? vrs : mrs, lane, q0 + z);
        cd[z] = load_offsets<I16>(irs, lane, q0 + z);
      }
  };
  const int first = pair0(0), first_cnt = nsl > 0 ? pair0(1) - first : 0;
  using StreamA = std::integral_constant<int, kStreamA>;
  using StreamM = std::integral_constant<int, PREC>; // A's own when there is none
  // One product: row j's sum of value * (gathered element of `src`, less
  // its own in difference form) is handed to finish(j, own, diagonal, sum).
  auto product = [&](auto stream, auto next, Rsrc src, auto own, auto diagonal, auto finish) {
    constexpr int S = decltype(stream)::value;
    using Acc = typename std::conditional<S == kStreamA, double, float>::type;
    constexpr bool DIFF = MIXED && S == kStreamA;
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        const int32_t row = row_of(j);
        const int q1 = pair0(j + 1);
        const T uv = own(j), gv = diagonal(j);
        Acc t0 = 0, t1 = 0;
        int c = pair0(j);
        do {
          const int cnt = q1 - c;
          T x0[CP], x1[CP];
#pragma unroll
          for (int z = 0; z < CP; ++z)
            if (z < cnt) {
              x0[z] = bload<T, kSc1>(src, row + cd[z].x());
              x1[z] = bload<T, kSc1>(src, row + cd[z].y());
            }
          V2 m[CP];
#pragma unroll
          for (int z = 0; z < CP; ++z)
            m[z] = cv[z];
          // the next chunk's loads go out before this chunk's gathers are used
          if (c + CP < q1)
            fetch(stream, c + CP, cnt - CP);
          else if (j + 1 < R && j + 1 < nsl)
            fetch(stream, q1, pair0(j + 2) - q1);
          else
            fetch(next, first, first_cnt);
#pragma unroll
          for (int z = 0; z < CP; ++z)
            if (z < cnt) {
              if constexpr (S == kStreamM16) { // two BF16 values in one word
                const uint32_t w = __float_as_uint(m[z].x);
                t0 += __uint_as_float(w << 16) * x0[z];
                t1 += __uint_as_float(w & 0xffff0000u) * x1[z];
              }
              else if constexpr (DIFF) { // padding: value 0, the row itself
                t0 += (Acc)m[z].x * ((Acc)x0[z] - (Acc)uv);
                t1 += (Acc)m[z].y * ((Acc)x1[z] - (Acc)uv);
              }
              else {
                t0 += m[z].x * x0[z];
                t1 += m[z].y * x1[z];
              }
            }
          c += CP;
        } while (c < q1);
        finish(j, uv, gv, t0 + t1);
      }
  };
  // u = M r from the published r; partials u.r and u.s
  auto precondition = [&](double (&v)[2]) {
    v[0] = v[1] = 0.0;
    product(
      StreamM{}, StreamA{}, rrs, [&](int j) { return (T)r[j]; },
      [&](int j) { return (T)bload<float, 0>(mds, row_of(j)); },
      [&](int j, T rv, T g, float t) {
        const float u = t + (float)g * (float)rv;
        di[DLDS ? 0 : j] = (T)u;
        bstore<float, kSc1>(urs, row_of(j), u);
        v[0] += (double)u * r[j];
        v[1] += (double)u * s[j];
      });
  };

  const int norm = a.norm;
  double rho = st.rho, beta = st.beta, rr_ref = st.rr_ref, rr_out = st.rr_out, tol2 = st.tol2;
  const double delta2 = st.delta2;
  const int max_iter = st.max_iter;
  int k = st.iter, nb_ru = st.nb_ru, converged = 0, breakdown = 0;
  const int k_end = k + a.max_launch_iter;
  bool finished = false;
  double* const keep = a.keep;

  if (!a.resume) {
    double v[3] = { 0.0, 0.0, 0.0 }; // r.u, r.r (or u.u), b.b
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        const double rd = residual(j), bd = bload<double, 0>(brs, row_of(j));
        r[j] = rd;
        if constexpr (FLEX) {
          bstore<T, kSc1>(rrs, row_of(j), (T)rd);
          v[1] += rd * rd;
          v[2] += bd * bd;
        }
        else {
          const T uv = get_u(j), mb = get_d(j) * (T)bd;
          bstore<T, kSc1>(urs, row_of(j), uv);
          v[0] += r[j] * (double)uv;
          v[1] += norm == 2 ? (double)uv * (double)uv : rd * rd;
          v[2] += norm == 2 ? (double)mb * (double)mb : bd * bd;
        }
      }
    if (!team_sum<3>(bar, v))
      return;
    tol2 = norm == 1 ? st.rtol2 * v[0] : fmax(st.rtol2 * v[2], st.atol2);
    rho = v[0];
    rr_ref = v[1];
    rr_out = v[1];
    beta = 0.0;
    finished = (norm == 1 ? v[0] : v[1]) <= tol2 || (!FLEX && v[0] == 0.0);
    converged = finished ? 1 : 0;
    if (me == 0 && threadIdx.x == 0) {
      st.bb = v[2];
      st.tol2 = tol2;
    }
  }
  else {
    const Rsrc krs = segment_buffer(keep, team.row0, rows);
    const Rsrc kps = segment_buffer(keep + a.n, team.row0, rows);
    const Rsrc kss = segment_buffer(keep + 2 * (int64_t)a.n, team.row0, rows);
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        r[j] = bload<double, 0>(krs, row_of(j));
        set_p(j, bload<double, 0>(kps, row_of(j)));
        s[j] = bload<double, 0>(kss, row_of(j));
        bstore<T, kSc1>(FLEX ? rrs : urs, row_of(j), FLEX ? (T)r[j] : get_u(j));
      }
    double v[1] = { 0.0 };
    if (!team_sum<1>(bar, v))
      return;
  }
  finished = finished || k >= max_iter;
  fetch(StreamM{}, first, first_cnt); // of A without a sparse preconditioner
  bool skip = FLEX;                   // a launch of the flexible method starts with u = M r

  while (!finished && k < k_end) {
    double alpha = 0.0;
    double v2[2] = { 0.0, 0.0 };
    bool updated = false; // a reliable update replaced r
    if (!skip) {
      // A
      double v1[1] = { 0.0 };
      product(
        StreamA{}, StreamM{}, urs, get_u, get_g,
        [&](int j, T uv, T g, double t) {
          const double pj = (double)uv + beta * get_p(j);
          set_p(j, pj);
          s[j] = (double)g * (double)uv + t + beta * s[j];
          v1[0] += pj * s[j];
        });
      if (!team_sum<1>(bar, v1))
        return;
      const double ps = v1[0];
      if (!(ps > 0.0) || !isfinite(ps) || (FLEX && !(rho > 0.0))) { // the operator is not positive definite on p
        breakdown = 1;
        finished = true;
        break;
      }
      // B
      alpha = rho / ps;
#pragma unroll
      for (int j = 0; j < R; ++j)
        if (j < nsl) {
          r[j] -= alpha * s[j];
          if constexpr (FLEX) {
            bstore<T, kSc1>(rrs, row_of(j), (T)r[j]);
            v2[1] += r[j] * r[j];
          }
          else {
            const T uv = get_u(j);
            bstore<T, kSc1>(urs, row_of(j), uv);
            v2[0] += r[j] * (double)uv;
            v2[1] += norm == 2 ? (double)uv * (double)uv : r[j] * r[j];
          }
          l_x[j * kBS] += alpha * get_p(j);
        }
      if (!team_sum<2>(bar, v2))
        return;
      const double rr = v2[1];
      if constexpr (MIXED) {
        if (rr <= delta2 * rr_ref || rr <= tol2 || k + 1 >= max_iter || !isfinite(rr)) {
          updated = true;
          publish_x();
          double v[1] = { 0.0 };
          if (!team_sum<1>(bar, v))
            return;
          v[0] = 0.0;
#pragma unroll
          for (int j = 0; j < R; ++j)
            if (j < nsl) {
              const double rd = residual(j);
              r[j] = rd;
              if constexpr (FLEX)
                bstore<T, kSc1>(rrs, row_of(j), (T)rd);
              v[0] += rd * rd;
            }
          if (!team_sum<1>(bar, v))
            return;
          ++nb_ru;
          rr_out = v[0];
          if (v[0] <= tol2 || k + 1 >= max_iter || !isfinite(v[0])) {
            converged = v[0] <= tol2 ? 1 : 0;
            ++k;
            finished = true;
            break;
          }
          rr_ref = v[0];
        }
        else
          rr_out = rr;
      }
    }
    if constexpr (FLEX) {
      double v[2];
      precondition(v);
      if (!team_sum<2>(bar, v))
        return;
      if (skip) {
        skip = false;
        if (!a.resume) { // else rho and beta come from the last launch
          rho = v[0];
          if (rho == 0.0) {
            finished = true;
            converged = 1;
          }
        }
        continue;
      }
      beta = updated ? v[0] / rho : -alpha * v[1] / rho;
      if (!(v[0] > 0.0) || !isfinite(v[0]) || !isfinite(beta)) { // M is not positive on this residual
        breakdown = 1;
        ++k;
        finished = true;
        break;
      }
      rho = v[0];
    }
    else {
      beta = rho != 0.0 ? v2[0] / rho : 0.0;
      rho = v2[0];
      if (updated) {
        double v[1] = { 0.0 };
#pragma unroll
        for (int j = 0; j < R; ++j)
          if (j < nsl) {
            const T uv = get_u(j);
            bstore<T, kSc1>(urs, row_of(j), uv);
            v[0] += r[j] * (double)uv;
          }
        if (!team_sum<1>(bar, v))
          return;
        rho = v[0];
      }
      if constexpr (!MIXED) {
        const double rr = v2[1], crit = norm == 1 ? rho : rr;
        rr_out = rr;
        if (crit <= tol2 || k + 1 >= max_iter || !isfinite(rr)) {
          converged = crit <= tol2 ? 1 : 0;
          ++k;
          finished = true;
          break;
        }
      }
    }
    ++k;
  }

  const bool lead = me == 0 && threadIdx.x == 0;
  if (finished) {
    publish_x();
    double v[1] = { 0.0 };
    if (!team_sum<1>(bar, v))
      return;
    v[0] = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        const double rd = residual(j);
        v[0] += rd * rd;
      }
    if (!team_sum<1>(bar, v))
      return;
    if (lead) {
      st.rr_true = v[0];
      st.done = 1;
      st.converged = converged;
    }
  }
  else {
    const Rsrc krs = segment_buffer(keep, team.row0, rows);
    const Rsrc kps = segment_buffer(keep + a.n, team.row0, rows);
    const Rsrc kss = segment_buffer(keep + 2 * (int64_t)a.n, team.row0, rows);
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        bstore<double, 0>(xrs, row_of(j), l_x[j * kBS]);
        bstore<double, 0>(krs, row_of(j), r[j]);
        bstore<double, 0>(kps, row_of(j), get_p(j));
        bstore<double, 0>(kss, row_of(j), s[j]);
      }
  }
  if (lead) {
    st.breakdown = breakdown;
    st.iter = k;
    st.nb_ru = nb_ru;
    st.rr_out = rr_out;
    st.rho = rho;
    st.beta = beta;
    st.rr_ref = rr_ref;
    st.epoch = bar.epoch;
  }
}

// Launches the kernel with room for `rows` slices per wave.
void launch_f64(const Args& a, int rows, bool idx16, int grid, size_t lds);
void launch_f32(const Args& a, int rows, bool idx16, int grid, size_t lds);
void launch_flex(const Args& a, int rows, bool idx16, bool bf16, int grid, size_t lds);

constexpr int kRowSteps[4] = { 1, 2, 5, 9 };

// 3x3 blocks (resident_block.hip): 512 threads, for 256 registers each.
constexpr int kBlockBS = 512;
constexpr int kBlockWaves = kBlockBS / kWave;
constexpr int kBlockRowSteps[3] = { 1, 2, 4 };
void launch_block(const Args& a, bool mixed, int rows, bool idx16, int grid);
void fill_block_values(const Pack& p, const int32_t* rp, const int32_t* ci, const double* v, bool want32);

template <class T, int PREC, bool I16>
inline void launch_kernel(const Args& a, int rows, int grid, size_t lds)
{
  auto go = [&](auto tag) {
    auto kernel = k_cg<T, decltype(tag)::value, I16, PREC>;
    AFEM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)lds));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBS), lds, stream(), a);
  };
  switch (rows) {
  case 1: go(std::integral_constant<int, 1>{}); break;
  case 2: go(std::integral_constant<int, 2>{}); break;
  case 5: go(std::integral_constant<int, 5>{}); break;
  default: go(std::integral_constant<int, 9>{}); break;
  }
  check_launch("resident_cg");
}

} // namespace resident
} // namespace afem
