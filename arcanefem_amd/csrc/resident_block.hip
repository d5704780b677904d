// resident_block.hip -- the resident conjugate-gradient kernel for systems of
// 3x3 blocks (three unknowns per node): the method, the barriers and the
// launch layout of resident_kernel.h, with a node in place of a row.
//
// Streams per node and iteration: FP32 14 blocks of 36 bytes and their
// offsets, once.  The gathers fetch a node's three numbers in one load and
// serve nine products each, so a wave keeps whole pairs of blocks in flight
// rather than many waves few: 512 threads of 256 registers a workgroup.  Bound
// by the stream (64 MB from the memory-side cache) and two barriers of 2.9 us.
// Block-Jacobi PCG, three kernels an iteration -> resident: 48 x 45 x 50 hexes
// of six tetrahedra (115 thousand nodes) mixed to 1e-8 1196 iterations of 30.3
// us -> 1060 of 16.4, with the copies of the values 37.2 -> 17.7 ms; the same
// in FP64 25.2 us an iteration; 9261 nodes mixed 8.7; 358 thousand nodes mixed
// 41.5, FP64 88 (4.5 TB/s).  Three pairs a chunk (two in FP64) spill at four
// nodes a lane: 43 and 127.
#include "resident_kernel.h"

namespace afem {
namespace resident {

typedef unsigned v3u __attribute__((ext_vector_type(3)));

// ---- numbers in pieces ------------------------------------------------------------------------
//
// N numbers per lane, stored as pieces of 16 bytes a lane (64 lanes next to
// each other) and a shorter last piece.

template <class T, int N>
__device__ __forceinline__ void store_pieces(T* base, int lane, const T (&m)[N])
{
  constexpr int PER = 16 / (int)sizeof(T), FULL = N / PER, REST = N % PER;
  typedef T VP __attribute__((ext_vector_type(PER)));
#pragma unroll
  for (int k = 0; k < FULL; ++k) {
    VP w;
#pragma unroll
    for (int c = 0; c < PER; ++c)
      w[c] = m[k * PER + c];
    *reinterpret_cast<VP*>(base + k * PER * kWave + lane * PER) = w;
  }
#pragma unroll
  for (int c = 0; c < REST; ++c)
    base[FULL * PER * kWave + lane * REST + c] = m[FULL * PER + c];
}

template <class T>
__device__ __forceinline__ void unpack4(T* m, v4u w)
{
  if constexpr (sizeof(T) == 4) {
    m[0] = __uint_as_float(w.x);
    m[1] = __uint_as_float(w.y);
    m[2] = __uint_as_float(w.z);
    m[3] = __uint_as_float(w.w);
  }
  else {
    m[0] = __longlong_as_double((long long)(((uint64_t)w.y << 32) | w.x));
    m[1] = __longlong_as_double((long long)(((uint64_t)w.w << 32) | w.z));
  }
}

// Group g of a buffer of groups of N numbers per lane.
template <class T, int N>
__device__ __forceinline__ void load_pieces(T (&m)[N], Rsrc r, int lane, int g)
{
  constexpr int PER = 16 / (int)sizeof(T), FULL = N / PER, REST = N % PER;
  constexpr int RB = REST * (int)sizeof(T); // bytes of the last piece: 0, 4 or 8
  const int at = g * (N * (int)sizeof(T) * kWave);
#pragma unroll
  for (int k = 0; k < FULL; ++k)
    unpack4<T>(m + k * PER, __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, at + k * (16 * kWave), 0));
  if constexpr (RB == 4)
    m[N - 1] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, at + FULL * (16 * kWave), 0));
  if constexpr (RB == 8) {
    const v2u w = __builtin_amdgcn_raw_buffer_load_b64(r, lane * 8, at + FULL * (16 * kWave), 0);
    if constexpr (sizeof(T) == 4) {
      m[N - 2] = __uint_as_float(w.x);
      m[N - 1] = __uint_as_float(w.y);
    }
    else
      m[N - 1] = __longlong_as_double((long long)(((uint64_t)w.y << 32) | w.x));
  }
}

// A node's three numbers.
template <class T, int AUX>
__device__ __forceinline__ void load3(T (&v)[3], Rsrc r, int32_t node)
{
  uint32_t off = (uint32_t)node * (uint32_t)(3 * sizeof(T));
  asm("" : "+v"(off)); // see bload
  if constexpr (sizeof(T) == 4) {
    const v3u w = __builtin_amdgcn_raw_buffer_load_b96(r, (int)off, 0, AUX);
    v[0] = __uint_as_float(w.x);
    v[1] = __uint_as_float(w.y);
    v[2] = __uint_as_float(w.z);
  }
  else {
    unpack4<double>(v, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, AUX));
    const v2u w = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 16, AUX);
    v[2] = __longlong_as_double((long long)(((uint64_t)w.y << 32) | w.x));
  }
}

template <class T, int AUX>
__device__ __forceinline__ void store3(Rsrc r, int32_t node, const T (&v)[3])
{
  const uint32_t off = (uint32_t)node * (uint32_t)(3 * sizeof(T));
  if constexpr (sizeof(T) == 4)
    __builtin_amdgcn_raw_buffer_store_b96(
      v3u{ __float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]) }, r, (int)off, 0, AUX);
  else {
    const uint64_t a = (uint64_t)__double_as_longlong(v[0]), b = (uint64_t)__double_as_longlong(v[1]),
                   c = (uint64_t)__double_as_longlong(v[2]);
    __builtin_amdgcn_raw_buffer_store_b128(
      v4u{ (uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32) }, r, (int)off, 0, AUX);
    __builtin_amdgcn_raw_buffer_store_b64(v2u{ (uint32_t)c, (uint32_t)(c >> 32) }, r, (int)off, 16, AUX);
  }
}

// ---- the kernel -------------------------------------------------------------------------------------

// Phases A and B and the mixed mode as in k_cg.  r, u, s and up to two nodes'
// D^-1 are in registers, x and p in LDS; in the mixed mode too r is FP64 and the
// terms of w are exact, differences and products (115 thousand nodes: FP64's
// 1060 iterations; differences rounded to FP32 1179, r as well 1273); the
// diagonal blocks (and D^-1 beyond two nodes a lane) come with the stream.
template <class T, int R, bool I16>
__global__ void __launch_bounds__(kBlockBS, 2) k_cg_block(Args a)
{
  using I2 = IndexPair<I16>;
  constexpr bool MIXED = sizeof(T) == 4;
  constexpr bool DREG = R <= (MIXED ? 2 : 1);
  constexpr int CP = MIXED ? 2 : 1; // pairs of a chunk
  extern __shared__ __align__(16) unsigned char smem[];

  const int wg = (int)xcd_tile(blockIdx.x, gridDim.x);
  const TeamDesc team = a.team[a.team_of[wg]];
  Status& st = a.st[team.seg];
  if (!st.active || st.done)
    return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int me = wg - team.wg0;

  const int64_t g0 = (int64_t)team.nslice * me / team.nwg, g1 = (int64_t)team.nslice * (me + 1) / team.nwg;
  const int s0 = (int)(g0 + (g1 - g0) * wave / kBlockWaves);
  const int nsl = (int)(g0 + (g1 - g0) * (wave + 1) / kBlockWaves) - s0;
  const int32_t po = a.poff[team.slice0 + s0 + min(lane, nsl)];
  auto pair0 = [&](int j) { return __builtin_amdgcn_readlane(po, j); };
  auto node_of = [&](int j) { return (s0 + j) * kWave + lane; };

  Barrier bar;
  bar.base = a.slots + (int64_t)team.wg0 * kSlotWords;
  bar.parity = (int64_t)gridDim.x * kSlotWords;
  bar.abort_flag = a.abort_flag;
  bar.limit = a.spin_limit;
  bar.me = me;
  bar.nwg = team.nwg;
  bar.epoch = st.epoch;

  const int32_t dofs = 3 * a.n;
  const Rsrc urs = segment_buffer(reinterpret_cast<const T*>(a.u), 0, dofs);
  const Rsrc xrs = segment_buffer(a.x, 0, dofs);
  const Rsrc brs = segment_buffer(a.b, 0, dofs);
  const Rsrc vrs = whole_buffer(a.v), irs = whole_buffer(a.idx);
  const Rsrc grs = whole_buffer(a.diag), drs = whole_buffer(a.dinv);

  double* l_x = reinterpret_cast<double*>(smem) + threadIdx.x; // [3][R], then p
  double* l_p = l_x + 3 * R * kBlockBS;
  T u[R][3], di[DREG ? R : 1][9];
  double r[R][3], s[R][3];
#pragma unroll
  for (int j = 0; j < R; ++j) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      u[j][c] = (T)0;
      r[j][c] = s[j][c] = 0.0;
      l_p[(3 * j + c) * kBlockBS] = 0.0;
    }
    if (j < nsl) {
      double xv[3];
      load3<double, 0>(xv, xrs, node_of(j));
#pragma unroll
      for (int c = 0; c < 3; ++c)
        l_x[(3 * j + c) * kBlockBS] = xv[c];
      if constexpr (DREG)
        load_pieces<T, 9>(di[j], drs, lane, s0 + j);
    }
  }

  auto mul9 = [](const auto (&m)[9], const auto (&v)[3], auto (&o)[3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      o[c] = m[3 * c] * v[0] + m[3 * c + 1] * v[1] + m[3 * c + 2] * v[2];
  };
  // D^-1 v of slice j
  auto jacobi = [&](int j, const double (&w)[3], T (&o)[3]) {
    const T v[3] = { (T)w[0], (T)w[1], (T)w[2] };
    if (!a.precond) {
#pragma unroll
      for (int c = 0; c < 3; ++c)
        o[c] = v[c];
    }
    else if constexpr (DREG)
      mul9(di[j], v, o);
    else {
      T d[9];
      load_pieces<T, 9>(d, drs, lane, s0 + j);
      mul9(d, v, o);
    }
  };

  // b - A64 x of slice j, x as published; 0 in the lanes past the last node
  auto residual = [&](int j, double (&rd)[3]) {
    const Rsrc v64 = whole_buffer(a.v64), g64 = whole_buffer(a.diag64);
    const int32_t node = node_of(j);
    double g[9], xv[3], bv[3], t[3];
    load_pieces<double, 9>(g, g64, lane, s0 + j);
    load3<double, 0>(bv, brs, node);
#pragma unroll
    for (int c = 0; c < 3; ++c)
      xv[c] = l_x[(3 * j + c) * kBlockBS];
    mul9(g, xv, t);
    const int q1 = pair0(j + 1);
    for (int q = pair0(j); q < q1; ++q) {
      double m[18], x0[3], x1[3];
      load_pieces<double, 18>(m, v64, lane, q);
      const I2 d = load_offsets<I16>(irs, lane, q);
      load3<double, kSc1>(x0, xrs, node + d.x());
      load3<double, kSc1>(x1, xrs, node + d.y());
#pragma unroll
      for (int c = 0; c < 3; ++c)
        t[c] += m[3 * c] * x0[0] + m[3 * c + 1] * x0[1] + m[3 * c + 2] * x0[2] + m[9 + 3 * c] * x1[0] +
                m[9 + 3 * c + 1] * x1[1] + m[9 + 3 * c + 2] * x1[2];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
      rd[c] = bv[c] - t[c];
  };
  auto publish_x = [&]() {
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        double xv[3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
          xv[c] = l_x[(3 * j + c) * kBlockBS];
        store3<double, kSc1>(xrs, node_of(j), xv);
      }
  };

  T cv[CP][18];
  I2 cd[CP];
  auto fetch = [&](int q0, int cnt) {
#pragma unroll
    for (int z = 0; z < CP; ++z)
      if (z < cnt) {
        load_pieces<T, 18>(cv[z], vrs, lane, q0 + z);
        cd[z] = load_offsets<I16>(irs, lane, q0 + z);
      }
  };
  const int first = pair0(0), first_cnt = nsl > 0 ? pair0(1) - first : 0;

  const int norm = a.norm;
  double rho = st.rho, beta = st.beta, rr_ref = st.rr_ref, rr_out = st.rr_out, tol2 = st.tol2;
  const double delta2 = st.delta2;
  const int max_iter = st.max_iter;
  int k = st.iter, nb_ru = st.nb_ru, converged = 0, breakdown = 0;
  const int k_end = k + a.max_launch_iter;
  bool finished = false;
  const Rsrc krs = segment_buffer(a.keep, 0, dofs);
  const Rsrc kps = segment_buffer(a.keep + dofs, 0, dofs);
  const Rsrc kss = segment_buffer(a.keep + 2 * (int64_t)dofs, 0, dofs);

  if (!a.resume) {
    double v[3] = { 0.0, 0.0, 0.0 }; // r.u, r.r (or u.u), b.b
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        double bd[3];
        T mb[3];
        residual(j, r[j]);
        load3<double, 0>(bd, brs, node_of(j));
        jacobi(j, r[j], u[j]);
        jacobi(j, bd, mb);
        store3<T, kSc1>(urs, node_of(j), u[j]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          v[0] += r[j][c] * (double)u[j][c];
          v[1] += norm == 2 ? (double)u[j][c] * (double)u[j][c] : r[j][c] * r[j][c];
          v[2] += norm == 2 ? (double)mb[c] * (double)mb[c] : bd[c] * bd[c];
        }
      }
    if (!team_sum<3, kBlockWaves>(bar, v))
      return;
    tol2 = norm == 1 ? st.rtol2 * v[0] : fmax(st.rtol2 * v[2], st.atol2);
    rho = v[0];
    rr_ref = v[1];
    rr_out = v[1];
    beta = 0.0;
    finished = (norm == 1 ? v[0] : v[1]) <= tol2 || v[0] == 0.0;
    converged = finished ? 1 : 0;
    if (me == 0 && threadIdx.x == 0) {
      st.bb = v[2];
      st.tol2 = tol2;
    }
  }
  else {
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        double pd[3];
        load3<double, 0>(r[j], krs, node_of(j));
        load3<double, 0>(pd, kps, node_of(j));
        load3<double, 0>(s[j], kss, node_of(j));
#pragma unroll
        for (int c = 0; c < 3; ++c)
          l_p[(3 * j + c) * kBlockBS] = pd[c];
        jacobi(j, r[j], u[j]);
        store3<T, kSc1>(urs, node_of(j), u[j]);
      }
    double v[1] = { 0.0 };
    if (!team_sum<1, kBlockWaves>(bar, v))
      return;
  }
  finished = finished || k >= max_iter;
  fetch(first, first_cnt);

  while (!finished && k < k_end) {
    // A
    double v1[1] = { 0.0 };
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        const int32_t node = node_of(j);
        const int q1 = pair0(j + 1);
        T g[9];
        load_pieces<T, 9>(g, grs, lane, s0 + j);
        double t[3] = { 0.0, 0.0, 0.0 };
        int q = pair0(j);
        do {
          const int cnt = q1 - q;
          T x0[CP][3], x1[CP][3];
#pragma unroll
          for (int z = 0; z < CP; ++z)
            if (z < cnt) {
              load3<T, kSc1>(x0[z], urs, node + cd[z].x());
              load3<T, kSc1>(x1[z], urs, node + cd[z].y());
            }
          T m[CP][18];
#pragma unroll
          for (int z = 0; z < CP; ++z)
#pragma unroll
            for (int e = 0; e < 18; ++e)
              m[z][e] = cv[z][e];
          // the next chunk's loads go out before this chunk's gathers are used
          if (q + CP < q1)
            fetch(q + CP, cnt - CP);
          else if (j + 1 < R && j + 1 < nsl)
            fetch(q1, pair0(j + 2) - q1);
          else
            fetch(first, first_cnt);
#pragma unroll
          for (int z = 0; z < CP; ++z)
            if (z < cnt) {
              double d0[3], d1[3]; // mixed: difference form; padding: value 0, the node itself
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                d0[c] = MIXED ? (double)x0[z][c] - (double)u[j][c] : (double)x0[z][c];
                d1[c] = MIXED ? (double)x1[z][c] - (double)u[j][c] : (double)x1[z][c];
              }
#pragma unroll
              for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                  t[c] = fma((double)m[z][3 * c + e], d0[e], t[c]);
                  t[c] = fma((double)m[z][9 + 3 * c + e], d1[e], t[c]);
                }
            }
          q += CP;
        } while (q < q1);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            t[c] = fma((double)g[3 * c + e], (double)u[j][e], t[c]);
          const double pj = (double)u[j][c] + beta * l_p[(3 * j + c) * kBlockBS];
          l_p[(3 * j + c) * kBlockBS] = pj;
          s[j][c] = t[c] + beta * s[j][c];
          v1[0] += pj * s[j][c];
        }
      }
    if (!team_sum<1, kBlockWaves>(bar, v1))
      return;
    const double ps = v1[0];
    if (!(ps > 0.0) || !isfinite(ps)) { // the operator is not positive definite on p
      breakdown = 1;
      finished = true;
      break;
    }
    // B
    const double alpha = rho / ps;
    double v2[2] = { 0.0, 0.0 };
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
          r[j][c] -= alpha * s[j][c];
        jacobi(j, r[j], u[j]);
        store3<T, kSc1>(urs, node_of(j), u[j]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          v2[0] += r[j][c] * (double)u[j][c];
          v2[1] += norm == 2 ? (double)u[j][c] * (double)u[j][c] : r[j][c] * r[j][c];
          l_x[(3 * j + c) * kBlockBS] += alpha * l_p[(3 * j + c) * kBlockBS];
        }
      }
    if (!team_sum<2, kBlockWaves>(bar, v2))
      return;
    const double rr = v2[1];
    beta = rho != 0.0 ? v2[0] / rho : 0.0;
    rho = v2[0];
    if constexpr (MIXED) {
      if (rr <= delta2 * rr_ref || rr <= tol2 || k + 1 >= max_iter || !isfinite(rr)) {
        // reliable update: r = b - A64 x
        publish_x();
        double v[1] = { 0.0 };
        if (!team_sum<1, kBlockWaves>(bar, v))
          return;
        v[0] = 0.0;
#pragma unroll
        for (int j = 0; j < R; ++j)
          if (j < nsl) {
            residual(j, r[j]);
#pragma unroll
            for (int c = 0; c < 3; ++c)
              v[0] += r[j][c] * r[j][c];
          }
        if (!team_sum<1, kBlockWaves>(bar, v))
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
        v[0] = 0.0;
#pragma unroll
        for (int j = 0; j < R; ++j)
          if (j < nsl) {
            jacobi(j, r[j], u[j]);
            store3<T, kSc1>(urs, node_of(j), u[j]);
#pragma unroll
            for (int c = 0; c < 3; ++c)
              v[0] += r[j][c] * (double)u[j][c];
          }
        if (!team_sum<1, kBlockWaves>(bar, v))
          return;
        rho = v[0];
      }
      else
        rr_out = rr;
    }
    else {
      const double crit = norm == 1 ? rho : rr;
      rr_out = rr;
      if (crit <= tol2 || k + 1 >= max_iter || !isfinite(rr)) {
        converged = crit <= tol2 ? 1 : 0;
        ++k;
        finished = true;
        break;
      }
    }
    ++k;
  }

  const bool lead = me == 0 && threadIdx.x == 0;
  if (finished) {
    publish_x();
    double v[1] = { 0.0 };
    if (!team_sum<1, kBlockWaves>(bar, v))
      return;
    v[0] = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        double rd[3];
        residual(j, rd);
#pragma unroll
        for (int c = 0; c < 3; ++c)
          v[0] += rd[c] * rd[c];
      }
    if (!team_sum<1, kBlockWaves>(bar, v))
      return;
    if (lead) {
      st.rr_true = v[0];
      st.done = 1;
      st.converged = converged;
    }
  }
  else {
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < nsl) {
        double xv[3], pd[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          xv[c] = l_x[(3 * j + c) * kBlockBS];
          pd[c] = l_p[(3 * j + c) * kBlockBS];
        }
        store3<double, 0>(xrs, node_of(j), xv);
        store3<double, 0>(krs, node_of(j), r[j]);
        store3<double, 0>(kps, node_of(j), pd);
        store3<double, 0>(kss, node_of(j), s[j]);
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

template <class T, bool I16>
static void launch(const Args& a, int rows, int grid)
{
  auto go = [&](auto tag) {
    constexpr int R = decltype(tag)::value;
    auto kernel = k_cg_block<T, R, I16>;
    const size_t lds = (size_t)R * kBlockBS * 48; // x and p
    AFEM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)lds));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlockBS), lds, stream(), a);
  };
  switch (rows) {
  case 1: go(std::integral_constant<int, 1>{}); break;
  case 2: go(std::integral_constant<int, 2>{}); break;
  default: go(std::integral_constant<int, 4>{}); break;
  }
  check_launch("resident_cg_block");
}

void launch_block(const Args& a, bool mixed, int rows, bool idx16, int grid)
{
  if (mixed && idx16)
    launch<float, true>(a, rows, grid);
  else if (mixed)
    launch<float, false>(a, rows, grid);
  else if (idx16)
    launch<double, true>(a, rows, grid);
  else
    launch<double, false>(a, rows, grid);
}

// ---- values -----------------------------------------------------------------------------------

// Blocks of a BSR matrix in pairs, the diagonal blocks and their inverses
// (adjugate / determinant; identity where that is zero or not finite), and
// (WANT32) the FP32 difference form.  Four waves a slice share its pairs; a
// lane reads its node's blocks where they lie (72 bytes each).  Bound by the
// copies' bytes (0.13 GB in, 0.19 GB out with FP32): 131 us at 115 thousand
// nodes, 2.4 TB/s, where the row sums and the two sliced copies of the
// streaming kernels take 500.
constexpr int kFillWaves = 4;

template <bool WANT32>
__global__ void __launch_bounds__(kFillWaves* kWave)
k_block_values(int32_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
               const double* __restrict__ v, const int32_t* __restrict__ poff, double* __restrict__ v64,
               double* __restrict__ diag64, double* __restrict__ dinv64, float* __restrict__ v32,
               float* __restrict__ diag32, float* __restrict__ dinv32)
{
  __shared__ double s_sum[kFillWaves][9][kWave];
  const int32_t s = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int32_t row = s * kWave + lane;
  const int32_t b = row < n ? rp[row] : 0, e = row < n ? rp[row + 1] : 0;
  double sum[9] = {};
  int32_t k = b;
  auto next = [&]() -> int32_t { // position of the row's next off-diagonal block
    while (k < e) {
      const int32_t at = k++;
      if (ci[at] != row)
        return at;
    }
    return -1;
  };
  const int64_t at = (int64_t)poff[s];
  const int w = poff[s + 1] - poff[s];
  for (int q = 0; q < w; ++q) {
    int2 f;
    f.x = next();
    f.y = next();
    if (q % kFillWaves != wave)
      continue;
    double m[18];
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      m[c] = f.x >= 0 ? v[9 * (int64_t)f.x + c] : 0.0;
      m[9 + c] = f.y >= 0 ? v[9 * (int64_t)f.y + c] : 0.0;
      sum[c] += m[c] + m[9 + c];
    }
    store_pieces<double, 18>(v64 + (at + q) * (18 * kWave), lane, m);
    if constexpr (WANT32) {
      float m32[18];
#pragma unroll
      for (int c = 0; c < 18; ++c)
        m32[c] = (float)m[c];
      store_pieces<float, 18>(v32 + (at + q) * (18 * kWave), lane, m32);
    }
  }
  if constexpr (WANT32) {
#pragma unroll
    for (int c = 0; c < 9; ++c)
      s_sum[wave][c][lane] = sum[c];
    __syncthreads();
  }
  if (wave != 0)
    return;
  double m[9] = {};
  bool has = false;
  for (int32_t z = b; z < e; ++z)
    if (ci[z] == row) {
      has = true;
#pragma unroll
      for (int c = 0; c < 9; ++c)
        m[c] += v[9 * (int64_t)z + c];
    }
  const int64_t d0 = (int64_t)s * (9 * kWave);
  store_pieces<double, 9>(diag64 + d0, lane, m);
  if constexpr (WANT32) {
    float g[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      double t = m[c];
      for (int q = 0; q < kFillWaves; ++q)
        t += s_sum[q][c][lane];
      g[c] = (float)t;
    }
    store_pieces<float, 9>(diag32 + d0, lane, g);
  }
  if (!has)
    m[0] = m[4] = m[8] = 1.0;
  double inv[9] = { m[4] * m[8] - m[5] * m[7], m[2] * m[7] - m[1] * m[8], m[1] * m[5] - m[2] * m[4],
                    m[5] * m[6] - m[3] * m[8], m[0] * m[8] - m[2] * m[6], m[2] * m[3] - m[0] * m[5],
                    m[3] * m[7] - m[4] * m[6], m[1] * m[6] - m[0] * m[7], m[0] * m[4] - m[1] * m[3] };
  const double det = m[0] * inv[0] + m[1] * inv[3] + m[2] * inv[6];
  const bool ok = det != 0.0 && isfinite(det);
  const double id = ok ? 1.0 / det : 1.0;
#pragma unroll
  for (int c = 0; c < 9; ++c)
    inv[c] = ok ? inv[c] * id : (c % 4 == 0 ? 1.0 : 0.0);
  store_pieces<double, 9>(dinv64 + d0, lane, inv);
  if constexpr (WANT32) {
    float i32[9];
#pragma unroll
    for (int c = 0; c < 9; ++c)
      i32[c] = (float)inv[c];
    store_pieces<float, 9>(dinv32 + d0, lane, i32);
  }
}

void fill_block_values(const Pack& p, const int32_t* rp, const int32_t* ci, const double* v, bool want32)
{
  if (want32)
    hipLaunchKernelGGL(k_block_values<true>, dim3(p.nslice), dim3(kFillWaves * kWave), 0, stream(), p.n, rp, ci, v,
                       p.poff.p, p.v64.p, p.diag64.p, p.dinv64.p, p.v32.p, p.diag32.p, p.dinv32.p);
  else
    hipLaunchKernelGGL(k_block_values<false>, dim3(p.nslice), dim3(kFillWaves * kWave), 0, stream(), p.n, rp, ci, v,
                       p.poff.p, p.v64.p, p.diag64.p, p.dinv64.p, (float*)nullptr, (float*)nullptr, (float*)nullptr);
}

} // namespace resident
} // namespace afem
