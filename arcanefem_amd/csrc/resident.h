// resident.h -- conjugate gradients of scalar systems and of systems of 3x3
// blocks in one launch: the vectors live in registers and LDS, the matrix in a
// pair layout read by wide loads, and the workgroups meet at barriers in
// device memory.
#pragma once

#include "common.h"

namespace afem {
namespace resident {

// Pair layout of a scalar matrix: slices of 64 rows; the off-diagonal entries
// of a row, in CSR order, fill pairs, and pair q of lane l of slice s is at
// (poff[s] + q) * 64 + l (values as two consecutive numbers, column offsets
// col - row as two consecutive 16- or 32-bit integers; padding: value 0,
// offset 0).  The diagonal entries are an array of their own.  Slices start
// at the first row of every segment.  With block = 3 rows and columns are
// nodes: a pair is two 3x3 blocks of 9 consecutive values, in pieces that a
// wave reads 64 x 16 bytes at a time, and the arrays of the diagonal hold
// blocks in the same kind of pieces, one per slice and lane.
struct Pack
{
  int block = 1;
  int32_t n = 0, nslice = 0, max_len = 0;
  int64_t npair = 0;
  bool idx16 = false;
  bool all_diag = false;            // every non-empty row has its diagonal entry
  std::vector<int32_t> seg_rows;    // row offsets of the segments
  std::vector<int32_t> seg_slices;  // first slice of each segment (nb_seg + 1)
  DBuf<int32_t> slice_row;          // per slice its first row, then the first and the end row of its segment
  DBuf<int32_t> poff;               // nslice + 1
  DBuf<int32_t> perm, inv;          // row of the matrix at each place, and back (empty: in order)
  DBuf<int32_t> src;                // with perm: 128 * npair positions in the CSR arrays (-1: padding)
  DBuf<int32_t> idx;                // 64 * npair (16-bit offsets) or 128 * npair words
  DBuf<double> v64, diag64, dinv64; // 128 * npair values; n (blocks: 9 times 128 * npair and 64 * nslice)
  DBuf<float> v32, diag32, dinv32;  // difference form: off-diagonal entries rounded, diag32 the row sum
  bool valid64 = false, valid32 = false;
  DBuf<uint32_t> m;                 // sparse preconditioner: 64 * npair words (BF16) or 128 * npair (FP32)
  DBuf<float> mdiag;
  int valid_prec = 0;               // 0, 16 or 32: the bits of the values in m
};

// Offsets of a pattern (rows rp, columns ci) cut into segments.  False: a
// segment alone does not fit the device, a column leaves its segment, or the
// layout pads too much.  `order` (device, may be null; one segment of scalar
// rows): a permutation of the rows by locality, used when neighbouring rows
// have unrelated columns.  block 3 (one segment): rows and columns of nodes,
// nnz blocks.
bool pack_pattern(Pack& p, int32_t n, int64_t nnz, const int32_t* rp, const int32_t* ci,
                  const std::vector<int32_t>& seg_rows, const int32_t* order = nullptr, int block = 1);
// Values of the pattern's matrix: FP64, and with want32 the FP32 difference form too.
void pack_values(Pack& p, const int32_t* rp, const int32_t* ci, const double* v, bool want32);

// Sparse preconditioner with the pattern's entries (v in CSR order), stored
// with 16 (BF16) or 32 bits.
void pack_prec(Pack& p, const int32_t* rp, const int32_t* ci, const float* v, int bits);

struct Status // of one segment
{
  double rtol2, atol2, delta2;      // in
  int max_iter, active;             // in; active 0: the segment is left alone
  double bb, tol2, rr_out, rr_true, rho, rr_ref, beta;
  int iter, done, converged, breakdown, nb_ru;
  unsigned epoch;                   // barriers taken since the slots were cleared
};

struct Options
{
  bool mixed = false;   // FP32 matrix and published vector, reliable updates in FP64
  bool precond = true;  // Jacobi
  int prec = 0;         // flexible CG with the pack's sparse preconditioner (its bits); mixed
  int norm = 0;         // stopping norm of afem_solver_options
  long long spin_limit = 0;
};

struct Round // segments that run together: one launch
{
  int first_word = 0; // of its teams in Work::team
  int teams = 0, grid = 0, rows_per_wave = 0;
  int64_t first_slot = 0;
};

// Work arrays kept by a solver: published vector, saved vectors, barrier slots.
struct Work
{
  DBuf<double> u;          // published vector (FP64, or FP32 in the same storage)
  DBuf<double> keep;       // r, p, s between launches
  DBuf<double> xb;         // x and b in the pack's order
  DBuf<uint64_t> slots;
  DBuf<int32_t> team;      // layout of the launches
  DBuf<Status> st;         // one per segment, then the abort flag
  Status* host = nullptr;  // pinned, nseg + 1
  int nseg = 0;
  unsigned epoch = 0;      // largest epoch in the slots
  std::vector<int32_t> layout_rows;
  std::vector<Round> rounds;
  void release() // the large arrays, when solves go another way
  {
    u.release();
    keep.release();
    xb.release();
    slots.release();
  }
  ~Work()
  {
    if (host)
      (void)hipHostFree(host);
  }
};

// run(), unless the memory for the layout, its values or the vectors is not
// there: then false, before anything was launched on x.
template <class F>
bool unless_out_of_memory(const F& run)
{
  try {
    return run();
  }
  catch (const Error& e) {
    if (e.status != AFEM_ERR_OUT_OF_MEMORY)
      throw;
    return false;
  }
}

// Runs the segments of w.host (inputs set, x the starting point) to their end;
// w.host holds the results.  False: a barrier wait gave up (x is then some
// iterate of each segment).
bool solve(const Pack& p, Work& w, const Options& o, double* x, const double* b);
// Launches that a solve of the pack's segments takes one after the other.
int round_count(const Pack& p);
// Makes room for the statuses of nseg segments.
void reserve(Work& w, int nseg);

} // namespace resident
} // namespace afem
