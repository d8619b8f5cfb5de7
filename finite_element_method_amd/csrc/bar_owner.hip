// bar_owner.hip -- one-pass assembly of truss and beam meshes.
//
// The host cuts the nodes into ranges of consecutive nodes.  Ranges whose
// nodes touch trusses only go to truss_owner_kernel (below: a compact entry
// record, rows 0..2 only); the others to bar_owner_kernel:
//
// One workgroup per range of owned nodes (<= 40 nodes, <= 256 incident
// (node, element) entries, <= 5120 CSR values).  Each element's constants (frame
// and term scales) sit in one 128-byte record, formed once per model change
// (bar_record_kernel) in the order in which the ranges meet the elements; an
// entry's block mask and row offsets are part of the pattern.  One lane per
// (owned node a, CSR row i) walks a's entries in element-insertion order and
// computes row i of each entry's global blocks (p, p) and (p, 1 - p) (p = a's
// position in the element).  The six lanes of a node sit in one wave and load
// each record together (16-byte loads), two entries ahead of the arithmetic,
// into the node's LDS slot,
// from which every lane reads it.  The diagonal block (a, a) is summed in
// registers over all incident elements (insertion order, starting from the
// first contribution); an off-diagonal block (a, b) has exactly one
// contributing element (checked when the maps are built).  The rows are formed
// in LDS and the workgroup's owned rows, one contiguous CSR range, are then
// written out by consecutive lanes as non-temporal 16-byte stores (a scattered
// row-by-row write costs one memory request per value).  Every CSR value is
// written once: no contribution buffer, no atomics, bitwise reproducible.
//
// Beam blocks use the rank-one form of beam.rs:495-605: with T = diag(R, R),
//   row i of T^T (sum_t s_t v_t,p v_t,q^T) T = sum_t s_t (T^T v_t,p)_i (T^T v_t,q)^T.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "device_state.hpp"
#include "element_math.hpp"
#include "fem_device.hpp"

namespace femdev {

namespace {

typedef double bo_d2 __attribute__((ext_vector_type(2)));

constexpr int BO_THREADS = 256;
constexpr int BO_NODES = 40;     // owned nodes per workgroup (10 per wave, 6 row lanes each)
constexpr int BO_ENTRIES = 256;  // (owned node, incident element) entries per workgroup
constexpr int BO_REC = 16;       // doubles per element record
constexpr int TO_REC = 6;        // truss kernel: doubles per element record (r, k_pp, k_pq, 0)
constexpr int BO_VALUES = 5120;  // CSR values of the owned rows per workgroup
constexpr int TO_NODES = 85;     // truss kernel: owned nodes per workgroup (3 row lanes each)
constexpr int TO_ENTRIES = 512;  // truss kernel: entries per workgroup

struct BarArgs {
  const double* __restrict__ xyz;
  const uint32_t* __restrict__ conn[2];
  const double* __restrict__ params[2];
  const double* __restrict__ R[2];
  const double* __restrict__ tdir;  // trusses: first rows of R, 3 doubles each
  const double* __restrict__ derived;
  const uint32_t* __restrict__ bid[2];
  const uint64_t* __restrict__ bmask;
  const uint16_t* __restrict__ boff;
  const uint32_t* __restrict__ inc_ptr;
  const uint32_t* __restrict__ inc;
  const uint2* __restrict__ ranges;  // per workgroup: first node, node count
  const double* __restrict__ rec;    // bar kernel: element records, BO_REC doubles each
  const uint32_t* __restrict__ entry_rec;  // entries, range r from entry_ptr[r]: type << 31 | record << 1 | p
  const uint32_t* __restrict__ entry_ptr;
  const uint4* __restrict__ entry;   // per entry: block (p, 1 - p); per node: its diagonal block (block_word)
  const uint4* __restrict__ self;
  const int64_t* __restrict__ row_ptr;
  double* __restrict__ val;
};

struct BarLds {
  uint32_t first[BO_NODES + 1];         // entry range of each owned node
  double2 slot[BO_NODES][BO_REC / 2 + 1];  // each owned node's current element record (padded: banks)
  uint4 block[BO_ENTRIES];              // the entries' off-diagonal blocks
  uint32_t rec[BO_ENTRIES];             // and their elements
  double out[BO_VALUES];                // the owned rows
};
static_assert(3 * sizeof(BarLds) <= 160 * 1024, "three workgroups per CU");

static_assert(BO_NODES == BAR_WG_NODES && BO_ENTRIES == BAR_WG_ENTRIES && BO_VALUES == BAR_WG_VALUES, "range cut");

// Truss-only ranges: rows 3..5 are empty and an entry needs five constants, so
// the layout is compact and a range holds up to twice the entries.
template <int ENTRIES, int VALUES>
struct TrussLds {
  double out[VALUES];          // the owned rows, one place in where their address is odd
  double data[ENTRIES][5];     // r (3), kpp, kpq
  uint4 block[ENTRIES];        // the entry's off-diagonal block
  uint8_t node[ENTRIES];       // owned node of the entry
  uint32_t first[TO_NODES + 1];
  uint32_t row[TO_NODES][3];   // start of rows 0..2 of each owned node, from the range's first value
};
constexpr int TO_STAGED = TRUSS_WG_STAGED;
static_assert(4 * sizeof(TrussLds<TO_STAGED, TRUSS_WG_VALUES + 2>) <= 160 * 1024, "four workgroups per CU");
static_assert(5 * sizeof(TrussLds<TO_ENTRIES, 2>) <= 160 * 1024, "five workgroups per CU");
static_assert(TO_STAGED <= BO_THREADS, "an entry per lane");
static_assert(TO_NODES == TRUSS_WG_NODES && TO_ENTRIES == TRUSS_WG_ENTRIES && 3 * TO_NODES <= BO_THREADS, "range cut");

// Jacobian of element e of `type` and the nodal shape derivatives b_p, b_q
// of its end p and the other end
__device__ inline double bar_shape(const BarArgs& A, int type, size_t e, int p, double& bp, double& bq) {
  const uint32_t n0 = A.conn[type][2 * e], n1 = A.conn[type][2 * e + 1];
  double d[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) d[k] = A.xyz[3 * size_t(n1) + k] - A.xyz[3 * size_t(n0) + k];
  const double Lg = fem::norm3(d[0], d[1], d[2]);
  const double J = fem::bar_jacobian(Lg);
  const double inv_j = 1.0 / J;
  bp = (p == 0 ? 0.0 - 0.5 : 0.0 + 0.5) * inv_j;
  bq = (p == 0 ? 0.0 + 0.5 : 0.0 - 0.5) * inv_j;
  return J;
}

// truss constants (truss.rs:132-189): direction r and the scales of the
// (p, p) and (p, q) blocks, k_pq = kpq r r^T
__device__ inline void truss_constants(const BarArgs& A, size_t e, int p, double o[5]) {
  double bp, bq;
  const double J = bar_shape(A, 0, e, p, bp, bq);
  const double* Rp = A.tdir + 3 * e;  // R's first row, stored compactly by the setup
  const double* prm = A.params[0] + 3 * e;
  const double E = prm[0], Ar = prm[1], A2 = prm[2];
  const double area = (A2 == A2) ? (A2 - Ar) / 2.0 * 0.0 + Ar - (A2 - Ar) / 2.0 * -1.0 : Ar;
  const double scale = area * E * J * 2.0;
  o[0] = Rp[0]; o[1] = Rp[1]; o[2] = Rp[2];
  o[3] = (bp * bp) * scale;
  o[4] = (bp * bq) * scale;
}

// An element's constants (beam: R (9), the scales of the rank-one terms u, v and
// w, tu, tv, tw, and |b_p|; truss: r (3), k_pp, k_pq; truss.rs:132-189,
// beam.rs:495-605).  One record serves both ends: with a copy per end (and the
// pattern's words in it, 160 bytes) the 64 x 64 x 64 frame holds 248 MB of
// constants, here 99 MB and 31 MB of entries.
__device__ inline void form_record(const BarArgs& A, uint32_t u, double* __restrict__ rec) {
  const int type = int(u >> 31);
  const size_t e = (u >> 1) & 0x3FFFFFFFu;
  double o[BO_REC];
#pragma unroll
  for (int k = 0; k < BO_REC; ++k) o[k] = 0.0;
  if (type == 0) {
    truss_constants(A, e, 0, o);  // k_pp and k_pq are the same from either end
  } else {
    double bp, bq;
    const double J = bar_shape(A, 1, e, 1, bp, bq);
    const double* Rp = A.R[1] + 9 * e;
    const double* prm = A.params[1] + 11 * e;
    const double E = prm[0], nu = prm[1], Ar = prm[2], it = prm[6], k = prm[7];
    const double G = E / (2.0 * (1.0 + nu));
    const double det_j = J, alpha = 2.0;
    const double i11p = A.derived[2 * e], i22p = A.derived[2 * e + 1];
#pragma unroll
    for (int m = 0; m < 9; ++m) o[m] = Rp[m];
    o[9] = Ar * E * det_j * alpha;
    o[10] = G * Ar * k * det_j * alpha;
    o[11] = G * it * det_j * alpha;
    o[12] = E * i22p * det_j * alpha;
    o[13] = E * i11p * det_j * alpha;
    o[14] = bp;  // of end 1; -bp exactly at end 0
    (void)bq;
  }
  double2* dst = reinterpret_cast<double2*>(rec);
#pragma unroll
  for (int k = 0; k < BO_REC / 2; ++k) dst[k] = make_double2(o[2 * k], o[2 * k + 1]);
}

// trusses of the truss kernel's ranges, formed in the same launch (blocks after the first n)
__device__ inline void form_truss_record(const BarArgs& A, uint32_t u, double* __restrict__ rec) {
  double o[TO_REC];
  o[5] = 0.0;
  truss_constants(A, (u >> 1) & 0x3FFFFFFFu, 0, o);
  double2* dst = reinterpret_cast<double2*>(rec);
#pragma unroll
  for (int k = 0; k < TO_REC / 2; ++k) dst[k] = make_double2(o[2 * k], o[2 * k + 1]);
}

__global__ __launch_bounds__(256) void bar_record_kernel(BarArgs A, const uint32_t* __restrict__ elem, size_t n,
                                                         double* __restrict__ rec,
                                                         const uint32_t* __restrict__ truss_elem, size_t n_truss,
                                                         double* __restrict__ truss_rec) {
  const size_t s = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (s < n) form_record(A, elem[s], rec + BO_REC * s);
  else if (s - n < n_truss) form_truss_record(A, truss_elem[s - n], truss_rec + TO_REC * (s - n));
}

// a block's mask (36 bits) and the offsets of its rows within the owned node's
// rows (12 bits each: a row holds at most 6 x 257 values)
__device__ inline uint4 block_word(const BarArgs& A, uint32_t k) {
  const uint64_t m = A.bmask[k];
  const uint16_t* o = A.boff + 6 * size_t(k);
  return make_uint4(uint32_t(m), uint32_t(m >> 32) | uint32_t(o[0]) << 4 | uint32_t(o[1]) << 16,
                    uint32_t(o[2]) | uint32_t(o[3]) << 12, uint32_t(o[4]) | uint32_t(o[5]) << 12);
}
__device__ inline uint32_t word_mask(const uint4& w, int i) {  // of row i
  return uint32_t((uint64_t(w.x) | uint64_t(w.y & 0xFu) << 32) >> (6 * i)) & 63u;
}
__device__ inline int word_off(const uint4& w, int i) {
  const uint32_t h = i < 2 ? w.y >> 4 : (i < 4 ? w.z : w.w);
  return int((i & 1 ? h >> 12 : h) & 0xFFFu);
}

// the entries' off-diagonal blocks, then the nodes' diagonal blocks (once per pattern)
__global__ __launch_bounds__(256) void bar_block_kernel(BarArgs A, const uint32_t* __restrict__ elem, size_t n_entries,
                                                        size_t n_nodes, uint4* __restrict__ entry,
                                                        uint4* __restrict__ self) {
  size_t s = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (s < n_entries) {
    const uint32_t u = A.entry_rec[s], type = u >> 31, p = u & 1u;
    const size_t e = (elem[(u >> 1) & 0x3FFFFFFFu] >> 1) & 0x3FFFFFFFu;
    entry[s] = block_word(A, A.bid[type][4 * e + 2 * p + (1 - p)]);
    return;
  }
  s -= n_entries;
  if (s >= n_nodes || A.inc_ptr[s] == A.inc_ptr[s + 1]) return;
  const uint32_t u = A.inc[A.inc_ptr[s]], p = u & 1u;
  self[s] = block_word(A, A.bid[u >> 31][4 * size_t((u >> 1) & 0x3FFFFFFFu) + 3 * p]);
}

// Row i = 3 h + m of an entry's blocks (p, p) -> self and (p, 1 - p) -> nb; o is
// the element's record, rec the same in LDS, from which a lane takes column m of
// R.  With v_t = T^T v_t,p the row is sum_t s_t v_t,i v_t in the order of t, where
//   u: (b r0, 0)  v: (b r1, -r2/2)  w: (b r2, -r1/2)  tu, tv, tw: (0, b r0..r2);
// products with those zeros are left out, and the other end's vectors (b turns
// its sign) share their products: 60 FP64 operations where the general sum over
// six-vectors took 110 and selected each v_t,i from six values.  This arithmetic
// bounded the kernel (64 x 64 x 64 frame: 125 -> 86 us; without the arithmetic 75).
__device__ inline void entry_rows(const double* __restrict__ o, const double* __restrict__ rec, uint32_t u, int h, int m,
                                  double self[6], double nb[6]) {
  const double x0 = rec[m];
  if (u >> 31 == 0) {  // truss: rows and columns 0..2
#pragma unroll
    for (int j = 0; j < 6; ++j) { self[j] = 0.0; nb[j] = 0.0; }
    if (h) return;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      self[j] = (x0 * o[3]) * o[j];
      nb[j] = (x0 * o[4]) * o[j];
    }
    return;
  }
  const double xv = rec[3 + 3 * h + m], xw = rec[6 - 3 * h + m];  // r1, r2 in a translation row; r2, r1 in a rotation row
  const double b = u & 1u ? o[14] : -o[14];
  const double bt = h ? 0.0 : b, br = h ? b : 0.0, bs = h ? -0.5 : b;
  const double su = o[9] * (bt * x0), sv = o[10] * (bs * xv), sw = o[10] * (bs * xw);
  const double s3 = o[11] * (br * x0), s4 = o[12] * (br * xw), s5 = o[13] * (br * xv);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const double b0 = b * o[j], b1 = b * o[3 + j], b2 = b * o[6 + j];
    const double t = __builtin_fma(sw, b2, __builtin_fma(sv, b1, su * b0));
    self[j] = t;
    nb[j] = -t;
    const double r = __builtin_fma(sw, -0.5 * o[3 + j], sv * (-0.5 * o[6 + j]));
    self[3 + j] = __builtin_fma(s5, b2, __builtin_fma(s4, b1, __builtin_fma(s3, b0, r)));
    nb[3 + j] = __builtin_fma(-s5, b2, __builtin_fma(-s4, b1, __builtin_fma(-s3, b0, r)));
  }
}

__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// row i of one block into the staged rows (r0: the row's start within them)
__device__ inline void write_row(BarLds& L, const uint4& w, int i, int r0, const double v[6]) {
  const uint32_t mi = word_mask(w, i);
  const int d0 = r0 + word_off(w, i);
#pragma unroll
  for (int j = 0; j < 6; ++j)
    if ((mi >> j) & 1u) L.out[d0 + __builtin_popcount(mi & ((1u << j) - 1u))] = v[j];
}

// One workgroup per range of owned nodes: one lane per (owned node, row) forms
// the rows in LDS, element records loaded two entries ahead; then consecutive
// lanes write the range out.  Bound: memory.  The 64 x 64 x 64 frame writes its
// 261 MB of values and reads 222 MB, of which 130 MB are records and entries
// once; the rest are those of elements whose other end lies in a range far away,
// read again.  98 us, 4.9 TB/s, the rate of a large copy (the compulsory bytes
// alone would take 66); called over and over on the same buffers, whose second
// reads the last-level cache then serves, 75 us.  LDS is busy 54 %, VALU 44 %.
__global__ __launch_bounds__(BO_THREADS) void bar_owner_kernel(BarArgs A) {
  __shared__ BarLds L;
  const int t = threadIdx.x;
  const uint2 rg = A.ranges[blockIdx.x];
  const uint32_t a0 = rg.x, na = rg.y;
  const uint32_t k0 = A.entry_ptr[blockIdx.x];
  const int ne = int(A.entry_ptr[blockIdx.x + 1] - k0);  // <= BO_ENTRIES (cut on the host)
  const uint32_t e0 = A.inc_ptr[a0];
  const int64_t base = A.row_ptr[6 * size_t(a0)];
  const int nv = int(A.row_ptr[6 * size_t(a0 + na)] - base);  // <= BO_VALUES (cut on the host)
  if (t < ne) {
    L.block[t] = A.entry[k0 + t];
    L.rec[t] = A.entry_rec[k0 + t];
  }
  if (t <= int(na)) L.first[t] = A.inc_ptr[a0 + t] - e0;
  __syncthreads();
  // lane (owned node j, row i), ten nodes per wave (lanes 60..63 idle here).
  // The six lanes of a node load one record together (lane i: 16-byte chunk i,
  // lanes 0 and 1 also chunks 6 and 7) into the node's LDS slot, and each reads
  // the whole record from there.
  const int jl = (t & 63) / 6, i = (t & 63) - 6 * jl;
  const int j = 10 * (t >> 6) + jl, h = i >= 3;
  if (jl < 10 && j < int(na)) {
    const size_t a = size_t(a0) + j;
    const int r0 = int(A.row_ptr[6 * a + i] - base);
    const bool row = A.row_ptr[6 * a + i + 1] - base > r0;
    const int s0 = int(L.first[j]), s1 = int(L.first[j + 1]);
    const uint4 diag = A.self[a];
    double2* __restrict__ buf = L.slot[j];
    const double2* __restrict__ recs = reinterpret_cast<const double2*>(A.rec);
    // chunks of the records one and two entries ahead
    double2 c0 = make_double2(0.0, 0.0), c1 = c0, f0 = c0, f1 = c0;
    auto load = [&](int sl, double2& x0, double2& x1) {
      if (sl >= s1) return;
      const double2* r = recs + (BO_REC / 2) * size_t((L.rec[sl] >> 1) & 0x3FFFFFFFu) + i;
      x0 = r[0];
      if (i < 2) x1 = r[6];
    };
    load(s0, c0, c1);
    load(s0 + 1, f0, f1);
    if (s1 > s0) {
      buf[i] = c0;
      if (i < 2) buf[6 + i] = c1;
    }
    wave_lds_sync();
    double acc[6];
    for (int sl = s0; sl < s1; ++sl) {
      c0 = f0;
      c1 = f1;
      load(sl + 2, f0, f1);
      double o[BO_REC];
#pragma unroll
      for (int m = 0; m < BO_REC / 2; ++m) {
        const double2 v = buf[m];
        o[2 * m] = v.x;
        o[2 * m + 1] = v.y;
      }
      if (row) {
        double self[6], nb[6];
        entry_rows(o, reinterpret_cast<const double*>(buf), L.rec[sl], h, i - 3 * h, self, nb);
#pragma unroll
        for (int q = 0; q < 6; ++q) acc[q] = sl == s0 ? self[q] : acc[q] + self[q];
        write_row(L, L.block[sl], i, r0, nb);
      }
      if (sl + 1 < s1) {
        wave_lds_sync();  // every lane of the node has read the slot
        buf[i] = c0;
        if (i < 2) buf[6 + i] = c1;
        wave_lds_sync();
      }
    }
    if (row && s1 > s0) write_row(L, diag, i, r0, acc);
  }
  __syncthreads();
  double* __restrict__ dst = A.val + base;
  // 16-byte stores from the first aligned address wherever the caller's array
  // starts, non-temporal (nothing in this kernel reads the values again); the odd
  // values at either end alone
  const int head = int((reinterpret_cast<uintptr_t>(dst) >> 3) & 1), npair = (nv - head) >> 1;
  for (int k = t; k < npair; k += BO_THREADS) {
    const int o = head + 2 * k;
    bo_d2 v;
    v.x = L.out[o];
    v.y = L.out[o + 1];
    __builtin_nontemporal_store(v, reinterpret_cast<bo_d2*>(dst + o));
  }
  if (t == 0 && head && nv > 0) dst[0] = L.out[0];
  if (t == BO_THREADS - 1 && nv > head && ((nv - head) & 1)) dst[nv - 1] = L.out[nv - 1];
}

// row i < 3 of a truss block (columns 0..2) straight to the CSR
__device__ inline void write_row3(double* val, const uint4& w, int i, int64_t r0, const double v[3]) {
  const uint32_t mi = word_mask(w, i) & 7u;
  double* dst = val + (r0 + word_off(w, i));
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if ((mi >> j) & 1u) dst[__builtin_popcount(mi & ((1u << j) - 1u))] = v[j];
}

// one truss entry (registers)
struct TrussEntry {
  double2 o[TO_REC / 2];
  uint4 block;
};
__device__ inline void truss_entry(const BarArgs& A, uint32_t k, TrussEntry& E) {
  const double2* r = reinterpret_cast<const double2*>(A.rec) + (TO_REC / 2) * size_t(A.entry_rec[k] >> 1);
  E.block = A.entry[k];
#pragma unroll
  for (int m = 0; m < TO_REC / 2; ++m) E.o[m] = r[m];
}
template <class Lds>
__device__ inline void put_entry(Lds& L, int sl, const TrussEntry& E) {
  L.data[sl][0] = E.o[0].x;
  L.data[sl][1] = E.o[0].y;
  L.data[sl][2] = E.o[1].x;
  L.data[sl][3] = E.o[1].y;
  L.data[sl][4] = E.o[2].x;
  L.block[sl] = E.block;
}

// Truss-only ranges: the same sums as bar_owner_kernel (diagonal block summed
// in insertion order from the first contribution, off-diagonal blocks written
// by their one element).  Entries come through 48-byte element records and the
// pattern's words, as the bar kernel's (a chain of look-ups per entry and 37 loads
// per wave before; launches back to back in a graph: 11 x 11 x 11 lattice 8.6 ->
// 4.95 us with the smaller ranges, 40 x 40 x 40 36.1 -> 29.5).  Whole calls of small
// meshes are bound by the host's part, 12.5 to 18 us from process to process.  An
// update of the areas forms the records anew, and with its assembly takes 32 us for
// the small lattice (49 before there were any) and 68 for the large.  Off-diagonal
// rows: one task per (row, entry), so that consecutive lanes write neighbouring
// blocks of one row.  Diagonal rows: one lane per (owned node, row 0..2).
//   STAGED: an entry per lane at most, rows staged in LDS and written as
//   16-byte chunks; four workgroups per CU (26 x 26 x 26 lattice 9.5 -> 8.7 us back
//   to back; 11 x 11 x 11 4.85 -> 4.95).
//   Otherwise rows straight to the CSR, five workgroups per CU; TWO: some range
//   has more entries than lanes, the loads of a lane's two in flight together.
template <bool TWO, bool STAGED>
__global__ __launch_bounds__(BO_THREADS) void truss_owner_kernel(BarArgs A) {
  __shared__ TrussLds<STAGED ? TO_STAGED : TO_ENTRIES, STAGED ? TRUSS_WG_VALUES + 2 : 2> L;
  const int t = threadIdx.x;
  const uint2 rg = A.ranges[blockIdx.x];
  const uint32_t a0 = rg.x, na = rg.y;
  const uint32_t e0 = A.inc_ptr[a0];
  const int ne = int(A.inc_ptr[a0 + na] - e0);  // <= TO_ENTRIES (cut on the host)
  const uint32_t k0 = A.entry_ptr[blockIdx.x];
  const int64_t base = A.row_ptr[6 * size_t(a0)];
  if (t <= int(na)) L.first[t] = A.inc_ptr[a0 + t] - e0;
  if (t < int(na)) {
    const int f0 = int(A.inc_ptr[a0 + t] - e0), f1 = int(A.inc_ptr[a0 + t + 1] - e0);
    for (int sl = f0; sl < f1; ++sl) L.node[sl] = uint8_t(t);
  }
  if (t < 3 * int(na)) L.row[t / 3][t % 3] = uint32_t(A.row_ptr[6 * size_t(a0 + t / 3) + t % 3] - base);
  if (ne > 0) {
    TrussEntry E0, E1;
    truss_entry(A, k0 + min(t, ne - 1), E0);
    if (TWO) truss_entry(A, k0 + min(t + BO_THREADS, ne - 1), E1);
    if (t < ne) put_entry(L, t, E0);
    if (TWO && t + BO_THREADS < ne) put_entry(L, t + BO_THREADS, E1);
  }
  __syncthreads();
  auto rows = [&](double* __restrict__ val) {
    for (int k = t; k < 3 * ne; k += BO_THREADS) {
      const int i = k / ne, sl = k - i * ne;
      const double* o = L.data[sl];
      const double s = o[i] * o[4];
      double nb[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) nb[q] = s * o[q];
      write_row3(val, L.block[sl], i, L.row[L.node[sl]][i], nb);
    }
    const int j = t / 3, i = t % 3;
    if (j >= int(na)) return;
    const int s0 = int(L.first[j]), s1 = int(L.first[j + 1]);
    if (s1 == s0) return;
    double acc[3];
    for (int sl = s0; sl < s1; ++sl) {
      const double* o = L.data[sl];
      const double s = o[i] * o[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) acc[q] = sl == s0 ? s * o[q] : acc[q] + s * o[q];
    }
    write_row3(val, A.self[a0 + j], i, L.row[j][i], acc);
  };
  double* __restrict__ dst = A.val + base;
  if (!STAGED) {
    rows(dst);
    return;
  }
  // staged from the parity of the address: pairs of values leave as aligned
  // 16-byte chunks wherever the caller's array starts, the odd values at either
  // end alone
  const int nv = int(A.row_ptr[6 * size_t(a0 + na)] - base);  // <= TRUSS_WG_VALUES (cut on the host)
  const int head = int((reinterpret_cast<uintptr_t>(dst) >> 3) & 1), npair = (nv - head) >> 1;
  double* const out = L.out + head;
  rows(out);
  __syncthreads();
  for (int k = t; k < npair; k += BO_THREADS) {
    const int o = head + 2 * k;
    bo_d2 v;
    v.x = out[o];
    v.y = out[o + 1];
    *reinterpret_cast<bo_d2*>(dst + o) = v;
  }
  if (t == 0 && head && nv > 0) dst[0] = out[0];
  if (t == BO_THREADS - 1 && nv > head && ((nv - head) & 1)) dst[nv - 1] = out[nv - 1];
}

}  // namespace

namespace {

BarArgs bar_args(Device* d, double* val) {
  BarArgs A;
  A.xyz = d->xyz;
  for (int t = 0; t < 2; ++t) {
    A.conn[t] = d->conn[t];
    A.params[t] = d->params[t];
    A.R[t] = d->R[t];
    A.bid[t] = d->bo_bid[t];
  }
  A.derived = d->derived;
  A.tdir = d->truss_dir;
  A.bmask = d->bo_bmask;
  A.boff = d->bo_boff;
  A.inc_ptr = d->bo_inc_ptr;
  A.inc = d->bo_inc;
  A.ranges = reinterpret_cast<const uint2*>(d->bo_ranges);
  A.rec = d->bo_rec;
  A.entry_rec = d->bo_entry_rec;
  A.entry_ptr = d->bo_entry_ptr;
  A.entry = d->bo_entry;
  A.self = d->bo_self;
  A.row_ptr = d->row_ptr;
  A.val = val;
  return A;
}

}  // namespace

// (re)forms the element records from the current coordinates, frames and
// parameters
std::string fill_bar_records(Device* d, hipStream_t s) {
  if (d->bo_n_recs + d->to_n_recs) {
    BarArgs A = bar_args(d, nullptr);
    bar_record_kernel<<<unsigned((d->bo_n_recs + d->to_n_recs + 255) / 256), 256, 0, s>>>(
        A, d->bo_rec_elem, d->bo_n_recs, d->bo_rec, d->to_rec_elem, d->to_n_recs, d->to_rec);
    HIP_TRY(hipGetLastError());
  }
  return "";
}

std::string upload_bar_maps(Device* d, const BarMaps& bm) {
  std::string e;
  for (int t = 0; t < 2; ++t)
    if (!(e = dupload(d->bo_bid[t], bm.bid[t].data(), bm.bid[t].size())).empty()) return e;
  if (!(e = dupload(d->bo_bmask, bm.bmask.data(), bm.bmask.size())).empty()) return e;
  if (!(e = dupload(d->bo_boff, bm.boff.data(), bm.boff.size())).empty()) return e;
  if (!(e = dupload(d->bo_inc_ptr, bm.inc_ptr.data(), bm.inc_ptr.size())).empty()) return e;
  if (!(e = dupload(d->bo_ranges, bm.ranges.data(), bm.ranges.size())).empty()) return e;
  d->bo_n_ranges = bm.n_bar_ranges;
  d->bo_n_truss_ranges = bm.ranges.size() / 2 - bm.n_bar_ranges;
  d->bo_truss_entries = 0;
  d->to_staged = bm.truss_staged;
  for (size_t r = bm.n_bar_ranges; r < bm.ranges.size() / 2; ++r)
    d->bo_truss_entries = std::max(d->bo_truss_entries, int(bm.inc_ptr[bm.ranges[2 * r] + bm.ranges[2 * r + 1]] -
                                                            bm.inc_ptr[bm.ranges[2 * r]]));
  if (!(e = dupload(d->bo_inc, bm.inc.data(), bm.inc.size())).empty()) return e;
  if (!(e = dupload(d->bo_rec_elem, bm.rec_elem.data(), bm.rec_elem.size())).empty()) return e;
  if (!(e = dupload(d->bo_entry_rec, bm.entry_rec.data(), bm.entry_rec.size())).empty()) return e;
  if (!(e = dupload(d->bo_entry_ptr, bm.entry_ptr.data(), bm.entry_ptr.size())).empty()) return e;
  d->bo_n_recs = bm.rec_elem.size();
  if (!(e = dupload(d->to_rec_elem, bm.truss_elem.data(), bm.truss_elem.size())).empty()) return e;
  if (!(e = dupload(d->to_entry_rec, bm.truss_entry.data(), bm.truss_entry.size())).empty()) return e;
  if (!(e = dupload(d->to_entry_ptr, bm.truss_ptr.data(), bm.truss_ptr.size())).empty()) return e;
  d->to_n_recs = bm.truss_elem.size();
  const size_t ne = bm.entry_rec.size(), nt = bm.truss_entry.size(), nn = ne + nt ? bm.inc_ptr.size() - 1 : 0;
  if (!(e = dalloc(d->bo_rec, size_t(BO_REC) * d->bo_n_recs)).empty()) return e;
  if (!(e = dalloc(d->bo_entry, ne)).empty()) return e;
  if (!(e = dalloc(d->bo_self, nn)).empty()) return e;
  if (!(e = dalloc(d->to_rec, size_t(TO_REC) * d->to_n_recs)).empty()) return e;
  if (!(e = dalloc(d->to_entry, nt)).empty()) return e;
  if (nn) {
    BarArgs A = bar_args(d, nullptr);
    bar_block_kernel<<<unsigned((ne + nn + 255) / 256), 256>>>(A, d->bo_rec_elem, ne, nn, d->bo_entry, d->bo_self);
    HIP_TRY(hipGetLastError());
    if (nt) {
      A.entry_rec = d->to_entry_rec;
      bar_block_kernel<<<unsigned((nt + 255) / 256), 256>>>(A, d->to_rec_elem, nt, 0, d->to_entry, d->bo_self);
      HIP_TRY(hipGetLastError());
    }
  }
  e = fill_bar_records(d, nullptr);
  if (!e.empty()) return e;
  d->kept = Kept::BAR_RECORDS;
  HIP_TRY(hipDeviceSynchronize());
  return "";
}

std::string assemble_bar_owner(Device* d, double* val, void* stream, bool timed) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (timed) HIP_TRY(hipEventRecord(d->ev0, s));
  if (d->bo_n_ranges + d->bo_n_truss_ranges) {
    BarArgs A = bar_args(d, val);
    if (d->bo_n_ranges) {
      bar_owner_kernel<<<unsigned(d->bo_n_ranges), BO_THREADS, 0, s>>>(A);
      HIP_TRY(hipGetLastError());
    }
    if (d->bo_n_truss_ranges) {
      A.ranges += d->bo_n_ranges;
      A.rec = d->to_rec;
      A.entry = d->to_entry;
      A.entry_rec = d->to_entry_rec;
      A.entry_ptr = d->to_entry_ptr;
      auto kernel = d->to_staged                      ? truss_owner_kernel<false, true>
                    : d->bo_truss_entries > BO_THREADS ? truss_owner_kernel<true, false>
                                                       : truss_owner_kernel<false, false>;
      kernel<<<unsigned(d->bo_n_truss_ranges), BO_THREADS, 0, s>>>(A);
      HIP_TRY(hipGetLastError());
    }
  }
  if (timed) {
    HIP_TRY(hipEventRecord(d->ev1, s));
    d->timed = true;
  }
  return "";
}

}  // namespace femdev
