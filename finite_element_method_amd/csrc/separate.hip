// separate.hip -- sparse partition of the assembled stiffness into K_aa, K_ab,
// K_ba, K_bb with k_aa_indexes, k_bb_indexes, r_a and u_b
// (methods_for_separate_stiffness_matrix.rs:217-345) on the device.
//
// A mask-and-compact over the CSR with no atomics and one wait of the host at the
// end.  Per row: its class (0 excluded: no stored diagonal or a zero one, 1 free
// = a, 2 constrained = b) and error; row positions by a scan of the classes;
// non-zero entries per row and target matrix; offsets by a scan of all four
// matrices' counts in one array; local columns and values, in column order, row
// pointers (rebased to 0 per matrix) and a summary in pinned host memory.
// Rows and columns of every output come out sorted.  The crate returns the
// first constrained dof without stiffness in index order: that is the minimum
// error key.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>
#include <string>

#include "device_state.hpp"
#include "fem_device.hpp"

namespace femdev {

namespace {

constexpr int SEP_SUMMARY = 12;  // err, n_aa, n_bb, nnz[4], entry offset[4], spare

template <class T>
std::string dgrow(T*& p, size_t& cap, size_t n) {
  if (n <= cap && p) return "";
  auto e = dalloc(p, n ? n : 1);
  if (!e.empty()) { cap = 0; return e; }
  cap = n ? n : 1;
  return "";
}

__device__ inline uint32_t lo32(uint64_t x) { return uint32_t(x); }
__device__ inline uint32_t hi32(uint64_t x) { return uint32_t(x >> 32); }

// G lanes per row (G a power of two <= 32): the lanes of a group stride over
// the row's entries together, so loads are coalesced; counts are combined
// with lane shuffles and output slots with wave ballots.  Every lane of a
// group has the same row, so groups enter and leave loops as a unit.
template <int G>
__device__ inline int group_sum(int x) {
  for (int o = G / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, G);
  return x;
}

// Position of each row's diagonal entry in the CSR (-1 when the pattern has
// none); depends on the pattern only, so it is computed once per pattern.
__global__ void sep_diag_pos(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci, int64_t n,
                             int64_t* __restrict__ dpos) {
  const int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r >= n) return;
  int64_t lo = rp[r], hi = rp[r + 1], found = -1;
  while (lo < hi) {  // columns ascend within a row
    const int64_t mid = (lo + hi) >> 1;
    const int64_t c = ci[mid];
    if (c == r) { found = mid; break; }
    if (c < r) lo = mid + 1; else hi = mid;
  }
  dpos[r] = found;
}

__global__ void sep_classify(const int64_t* __restrict__ dpos, const double* __restrict__ val,
                             const uint8_t* __restrict__ cons, int64_t n, uint8_t* __restrict__ cls,
                             uint64_t* __restrict__ flag, int64_t* __restrict__ key, int64_t* __restrict__ cnt) {
  const int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r > n) return;
  if (r == n) {  // totals slot of the scans
    flag[n] = 0;
    cnt[2 * n] = 0;
    return;
  }
  const int64_t p = dpos[r];
  const double diag = p >= 0 ? val[p] : 0.0;
  const bool c_r = cons[r] != 0;
  const uint8_t k = diag == 0.0 ? 0 : (c_r ? 2 : 1);
  cls[r] = k;
  flag[r] = uint64_t(k == 1) | (uint64_t(k == 2) << 32);
  key[r] = (diag == 0.0 && c_r) ? r : INT64_MAX;
  cnt[2 * r] = 0;
  cnt[2 * r + 1] = 0;
}

// Row-count slots: K_aa rows at [0, na), K_ab at [na, 2na), K_ba at
// [2na, 2na + nb), K_bb at [2na + nb, 2na + 2nb).
template <int G>
__global__ void sep_count(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                          const double* __restrict__ val, const uint8_t* __restrict__ cls,
                          const uint64_t* __restrict__ pos, const double* __restrict__ force,
                          const double* __restrict__ disp, int64_t n, int64_t* __restrict__ cnt,
                          int64_t* __restrict__ aa_idx, int64_t* __restrict__ bb_idx, double* __restrict__ r_a,
                          double* __restrict__ u_b) {
  const int64_t r = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / G;
  const int lig = threadIdx.x & (G - 1);
  if (r >= n) return;
  const uint8_t k = cls[r];
  if (k == 0) return;
  int ca = 0, cb = 0;
  for (int64_t e = rp[r] + lig; e < rp[r + 1]; e += G) {
    if (val[e] == 0.0) continue;
    const uint8_t kc = cls[ci[e]];
    ca += kc == 1;
    cb += kc == 2;
  }
  ca = group_sum<G>(ca);
  cb = group_sum<G>(cb);
  if (lig != 0) return;
  const int64_t na = lo32(pos[n]), nb = hi32(pos[n]);
  if (k == 1) {
    const int64_t pa = lo32(pos[r]);
    cnt[pa] = ca;
    cnt[na + pa] = cb;
    aa_idx[pa] = r;
    r_a[pa] = force[r];
  } else {
    const int64_t pb = hi32(pos[r]);
    cnt[2 * na + pb] = ca;
    cnt[2 * na + nb + pb] = cb;
    bb_idx[pb] = r;
    u_b[pb] = disp[r];
  }
}

template <int G>
__global__ void sep_fill(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                         const double* __restrict__ val, const uint8_t* __restrict__ cls,
                         const uint64_t* __restrict__ pos, const int64_t* __restrict__ off, int64_t n,
                         int32_t* __restrict__ out_ci, double* __restrict__ out_v) {
  const int64_t r = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / G;
  const int lane = threadIdx.x & 63, lig = threadIdx.x & (G - 1);
  if (r >= n) return;
  const uint8_t k = cls[r];
  if (k == 0) return;
  const int64_t na = lo32(pos[n]), nb = hi32(pos[n]);
  int64_t o_a, o_b;  // next slot of an entry in an a column / a b column
  if (k == 1) {
    const int64_t pa = lo32(pos[r]);
    o_a = off[pa];
    o_b = off[na + pa];
  } else {
    const int64_t pb = hi32(pos[r]);
    o_a = off[2 * na + pb];
    o_b = off[2 * na + nb + pb];
  }
  const uint64_t group = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << (lane & ~(G - 1));
  const uint64_t below = (1ull << lane) - 1ull;
  const int64_t end = rp[r + 1];
  for (int64_t base = rp[r]; base < end; base += G) {
    const int64_t e = base + lig;
    double v = 0.0;
    int32_t c = 0;
    uint8_t kc = 0;
    if (e < end) {
      v = val[e];
      c = ci[e];
      if (v != 0.0) kc = cls[c];
    }
    const uint64_t ba = __ballot(kc == 1) & group, bb = __ballot(kc == 2) & group;
    if (kc == 1) {
      const int64_t o = o_a + __popcll(ba & below);
      out_ci[o] = int32_t(lo32(pos[c]));
      out_v[o] = v;
    } else if (kc == 2) {
      const int64_t o = o_b + __popcll(bb & below);
      out_ci[o] = int32_t(hi32(pos[c]));
      out_v[o] = v;
    }
    o_a += __popcll(ba);
    o_b += __popcll(bb);
  }
}

// ---- four values per lane (values under 4 GiB, the default)
//
//   values   per row its non-zero entries and its class (reads the values only)
//   classes  a and b dofs per SEP_CHUNK dofs, and the first error
//   chunks   their exclusive sums (one workgroup)
//   pack     per dof one word, class << 30 | its index among the a (or b) dofs;
//            the index lists, r_a and u_b
//   mark     the rows that hold a column that is not free.  The pattern is
//            symmetric, so these are the columns of the rows that are not free:
//            few, as a rule
//   count    the entries of marked rows in a columns and in b columns (an unmarked
//            row's all go to a columns), and per SEP_ROWS rows and target matrix
//            their sums
//   scan     the sums of all four matrices in one array: the matrices follow each
//            other in the output
//   fill     row offsets from the counts, row pointers, local columns and values:
//            runs of rows that go to K_aa as they are, then the other rows
//
// Bound: memory.  The fill reads and writes 12 bytes per entry, the first pass
// reads 8.
constexpr uint32_t SEP_IDX = (1u << 30) - 1u;
constexpr int SEP_CHUNK = 1024;  // dofs per workgroup of classes and pack, four per thread
// Few restrained dofs: at most one in this many.  A restrained dof marks the 20
// to 40 rows of its neighbours; past that share most rows are marked, and the
// first pass over the values alone is lost: with 5 % of the dofs restrained at
// random 592 us, against 453 with the classes from the diagonals and one count with
// columns (512 x 512 plate; a restrained edge, 0.2 %: 293 us).
constexpr int SEP_FEW = 128;
constexpr int SEP_ROWS = 64;     // rows per wave of values, mark, count and fill
typedef unsigned int sep_u32x4 __attribute__((ext_vector_type(4)));

// bytes 4 t .. 4 t + 3 of an array of n bytes (0 past its end)
__device__ inline uint32_t load_bytes4(const uint8_t* __restrict__ a, int64_t i, int64_t n) {
  if (i + 4 <= n) return *reinterpret_cast<const uint32_t*>(a + i);
  uint32_t w = 0;
  for (int k = 0; k < 4; ++k)
    if (i + k < n) w |= uint32_t(a[i + k]) << (8 * k);
  return w;
}
// inclusive sum over a wave
template <class T>
__device__ inline T wave_scan(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T u = __shfl_up(v, o);
    if (lane >= o) v += u;
  }
  return v;
}

// exclusive sum over a workgroup of W waves, and the total
template <int W>
__device__ inline uint64_t block_scan(uint64_t v, uint64_t& total) {
  __shared__ uint64_t w[W];
  const uint64_t incl = wave_scan(v);
  if ((threadIdx.x & 63) == 63) w[threadIdx.x >> 6] = incl;
  __syncthreads();
  uint64_t before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < W; ++k) {
    if (k < int(threadIdx.x >> 6)) before += w[k];
    all += w[k];
  }
  __syncthreads();  // w may be written again
  total = all;
  return before + incl - v;
}

__device__ inline void sep_values4(__amdgpu_buffer_rsrc_t rv, uint32_t e, double w[4]) {
  const double2 w0 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * e, 0, 0));
  const double2 w1 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * e + 16u, 0, 0));
  w[0] = w0.x; w[1] = w0.y; w[2] = w1.x; w[3] = w1.y;
}
__device__ inline void sep_columns4(__amdgpu_buffer_rsrc_t rc, uint32_t e, uint32_t c[4]) {
  const sep_u32x4 cc = __builtin_amdgcn_raw_buffer_load_b128(rc, 4u * e, 0, 0);
  c[0] = cc.x; c[1] = cc.y; c[2] = cc.z; c[3] = cc.w;
}

// A wave per SEP_ROWS rows, 16 at a time, four lanes per row, each taking four
// neighbouring entries per step with two 16-byte loads (range-checked: entries
// past a row are loaded but not used).  The diagonal, whose value gives the
// class, passes by among the row's values (gathered on its own it cost as many
// lines as rows).
__global__ __launch_bounds__(256) void sep_values(const int64_t* __restrict__ rp, const int64_t* __restrict__ dpos,
                                                  const double* __restrict__ val, const uint8_t* __restrict__ cons,
                                                  int64_t n, uint2* __restrict__ counts, uint8_t* __restrict__ cls,
                                                  uint8_t* __restrict__ mark, uint32_t v_bytes) {
  const int lane = threadIdx.x & 63, lig = lane & 3;
  const int64_t r0 = (int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * SEP_ROWS;
  if (r0 >= n) return;
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(val), 0, int(v_bytes), 0x00020000);
  const int64_t r = r0 + lane;  // the lane's own row
  const bool on = r < n;
  const uint32_t start = on ? uint32_t(rp[r]) : 0u, end = on ? uint32_t(rp[r + 1]) : 0u;
  const int64_t dp = on ? dpos[r] : -1;
  const uint32_t diag = dp < 0 ? 0xFFFFFFFFu : uint32_t(dp);
  uint32_t total = 0;
  bool zero = true;
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    const int src = 16 * pass + (lane >> 2);
    const uint32_t b = uint32_t(__shfl(int(start), src)), q = uint32_t(__shfl(int(end), src)),
                   di = uint32_t(__shfl(int(diag), src));
    uint32_t c = 0;
    int nz = 0;  // the diagonal is stored and not zero
    for (uint32_t e = b + 4u * lig; e < q; e += 16u) {
      double w[4];
      sep_values4(rv, e, w);
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const bool x = e + j < q && w[j] != 0.0;
        c += x;
        nz |= x && e + j == di;
      }
    }
#pragma unroll
    for (int o = 2; o > 0; o >>= 1) {
      c += uint32_t(__shfl_xor(int(c), o, 4));
      nz |= __shfl_xor(nz, o, 4);
    }
    // row `src` sits in lanes 4 (lane >> 2) ..: hand it to its own lane
    const uint32_t cc = uint32_t(__shfl(int(c), 4 * (lane & 15)));
    const int zz = __shfl(nz, 4 * (lane & 15));
    if ((lane >> 4) == pass) {
      total = cc;
      zero = zz == 0;
    }
  }
  if (!on) return;
  counts[r] = make_uint2(total, 0u);
  cls[r] = uint8_t(zero ? 0 : (cons[r] ? 2 : 1));
  mark[r] = 0;
}

// class of each dof from its diagonal's value alone (many restrained dofs: the
// rows are counted with their columns later)
__global__ __launch_bounds__(256) void sep_diagonals(const int64_t* __restrict__ dpos, const double* __restrict__ val,
                                                     const uint8_t* __restrict__ cons, int64_t n,
                                                     uint8_t* __restrict__ cls) {
  const int64_t r = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (r >= n) return;
  const int64_t p = dpos[r];
  const bool zero = p < 0 || val[p] == 0.0;
  cls[r] = uint8_t(zero ? 0 : (cons[r] ? 2 : 1));
}

__global__ __launch_bounds__(256) void sep_classes(const uint8_t* __restrict__ cls, const uint8_t* __restrict__ cons,
                                                   int64_t n, uint64_t* __restrict__ chunk,
                                                   uint32_t* __restrict__ chunk_err) {
  __shared__ uint32_t err[4];
  const int64_t r0 = int64_t(blockIdx.x) * SEP_CHUNK + 4 * threadIdx.x;
  const uint32_t k4 = r0 < n ? load_bytes4(cls, r0, n) : 0u, c4 = r0 < n ? load_bytes4(cons, r0, n) : 0u;
  uint32_t bad = 0xFFFFFFFFu, na = 0, nb = 0;
#pragma unroll
  for (int k = 3; k >= 0; --k) {
    const uint32_t kk = (k4 >> (8 * k)) & 255u;
    na += kk == 1u;
    nb += kk == 2u;
    if (kk == 0u && ((c4 >> (8 * k)) & 255u)) bad = uint32_t(r0) + k;  // constrained, without stiffness
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) bad = min(bad, uint32_t(__shfl_xor(int(bad), o)));
  if ((threadIdx.x & 63) == 0) err[threadIdx.x >> 6] = bad;
  uint64_t total;
  block_scan<4>(uint64_t(na) | uint64_t(nb) << 32, total);  // its barriers order err, too
  if (threadIdx.x == 0) {
    chunk[blockIdx.x] = total;
    chunk_err[blockIdx.x] = min(min(err[0], err[1]), min(err[2], err[3]));
  }
}

// head: the first error row (INT64_MAX: none), n_aa, n_bb
__global__ __launch_bounds__(1024) void sep_chunks(uint64_t* __restrict__ chunk, const uint32_t* __restrict__ chunk_err,
                                                   int n_chunks, int64_t* __restrict__ head) {
  __shared__ uint32_t err[16];
  uint64_t sum = 0;
  uint32_t bad = 0xFFFFFFFFu;
  for (int b = 0; b < n_chunks; b += 1024) {
    const int i = b + int(threadIdx.x);
    uint64_t total;
    const uint64_t before = block_scan<16>(i < n_chunks ? chunk[i] : 0ull, total);
    if (i < n_chunks) {
      chunk[i] = sum + before;
      bad = min(bad, chunk_err[i]);
    }
    sum += total;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) bad = min(bad, uint32_t(__shfl_xor(int(bad), o)));
  if ((threadIdx.x & 63) == 0) err[threadIdx.x >> 6] = bad;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 16; ++k) bad = min(bad, err[k]);
    head[0] = bad == 0xFFFFFFFFu ? INT64_MAX : int64_t(bad);
    head[1] = int64_t(lo32(sum));
    head[2] = int64_t(hi32(sum));
  }
}

__global__ __launch_bounds__(256) void sep_pack_rows(const uint8_t* __restrict__ cls, const uint64_t* __restrict__ chunk,
                                                     const double* __restrict__ force, const double* __restrict__ disp,
                                                     int64_t n, uint32_t* __restrict__ pack,
                                                     int64_t* __restrict__ aa_idx, int64_t* __restrict__ bb_idx,
                                                     double* __restrict__ r_a, double* __restrict__ u_b) {
  const int64_t r0 = int64_t(blockIdx.x) * SEP_CHUNK + 4 * threadIdx.x;
  const uint32_t k4 = r0 < n ? load_bytes4(cls, r0, n) : 0u;
  uint32_t na = 0, nb = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    na += ((k4 >> (8 * k)) & 255u) == 1u;
    nb += ((k4 >> (8 * k)) & 255u) == 2u;
  }
  uint64_t total;
  const uint64_t at = chunk[blockIdx.x] + block_scan<4>(uint64_t(na) | uint64_t(nb) << 32, total);
  uint32_t a = lo32(at), b = hi32(at), w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t kk = (k4 >> (8 * k)) & 255u;
    w[k] = kk == 0u ? 0u : kk << 30 | (kk == 1u ? a : b);
    if (kk == 1u) {
      aa_idx[a] = r0 + k;
      r_a[a] = force[r0 + k];
      ++a;
    } else if (kk == 2u) {
      bb_idx[b] = r0 + k;
      u_b[b] = disp[r0 + k];
      ++b;
    }
  }
  if (r0 + 4 <= n) {
    *reinterpret_cast<uint4*>(pack + r0) = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
    for (int k = 0; k < 4; ++k)
      if (r0 + k < n) pack[r0 + k] = w[k];
  }
}

// a wave per SEP_ROWS rows: it takes the rows that are not free one after
// another, their columns over its lanes
__global__ __launch_bounds__(256) void sep_mark(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                const uint8_t* __restrict__ cls, int64_t n, uint8_t* __restrict__ mark) {
  const int lane = threadIdx.x & 63;
  const int64_t r0 = (int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * SEP_ROWS;
  const int64_t r = r0 + lane;
  uint64_t todo = __ballot(r < n && cls[r < n ? r : 0] != 1);
  while (todo) {
    const int64_t q = r0 + __builtin_ctzll(todo);
    todo &= todo - 1;
    for (int64_t e = rp[q] + lane; e < rp[q + 1]; e += 64) mark[ci[e]] = 1;  // any writer stores the same
  }
}

// the group's sums per target matrix, from a row's class and counts per lane
__device__ inline void put_sums(uint32_t k, uint2 c, int lane, int64_t g, int64_t* __restrict__ sums, int64_t n_groups) {
  uint32_t s[4] = {k == 1u ? c.x : 0u, k == 1u ? c.y : 0u, k == 2u ? c.x : 0u, k == 2u ? c.y : 0u};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s[w] += uint32_t(__shfl_xor(int(s[w]), o));
    if (lane == w) sums[int64_t(w) * n_groups + g] = int64_t(s[w]);
  }
  if (g == 0 && lane == 0) sums[4 * n_groups] = 0;  // totals slot of the scan
}

// A wave per SEP_ROWS rows, a lane per row; where there are marked rows, eight
// rows at a time with eight lanes each.  sums: at w * n_groups + group the
// entries of its rows in matrix w.
__global__ __launch_bounds__(256) void sep_count_rows(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                      const double* __restrict__ val, const uint32_t* __restrict__ pack,
                                                      const uint8_t* __restrict__ mark, int64_t n,
                                                      uint2* __restrict__ counts, int64_t* __restrict__ sums,
                                                      int64_t n_groups) {
  const int lane = threadIdx.x & 63;
  const int64_t g = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (g >= n_groups) return;
  const int64_t r = g * SEP_ROWS + lane;
  const uint32_t k = r < n ? pack[r] >> 30 : 0u;
  uint2 c = k ? counts[r] : make_uint2(0u, 0u);
  const uint64_t marked = __ballot(k != 0u && mark[k ? r : 0] != 0);
#pragma unroll 1
  for (int pass = 0; pass < SEP_ROWS / 8; ++pass) {
    if (!((marked >> (8 * pass)) & 255ull)) continue;
    const int row = 8 * pass + (lane >> 3);
    const int64_t q = g * SEP_ROWS + row;
    uint32_t ca = 0, cb = 0;
    if ((marked >> row) & 1ull)
      for (int64_t e = rp[q] + (lane & 7); e < rp[q + 1]; e += 8)
        if (val[e] != 0.0) {
          const uint32_t kc = pack[ci[e]] >> 30;
          ca += kc == 1u;
          cb += kc == 2u;
        }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) {
      ca += uint32_t(__shfl_xor(int(ca), o, 8));
      cb += uint32_t(__shfl_xor(int(cb), o, 8));
    }
    // the row's sums from its eight lanes to its own lane
    const uint32_t sa = uint32_t(__shfl(int(ca), 8 * (lane & 7))), sb = uint32_t(__shfl(int(cb), 8 * (lane & 7)));
    if ((lane >> 3) == pass && ((marked >> lane) & 1ull)) {
      c = make_uint2(sa, sb);
      counts[r] = c;
    }
  }
  put_sums(k, c, lane, g, sums, n_groups);
}

// the same with every row's columns read: a workgroup per SEP_ROWS rows, four
// lanes per row, four neighbouring entries per lane and step
constexpr int SEP_QL_COUNT = 4;
__global__ __launch_bounds__(SEP_ROWS* SEP_QL_COUNT) void sep_count_all(
    const int64_t* __restrict__ rp, const int32_t* __restrict__ ci, const double* __restrict__ val,
    const uint32_t* __restrict__ pack, int64_t n, uint2* __restrict__ counts, int64_t* __restrict__ sums,
    int64_t n_groups, uint32_t v_bytes) {
  __shared__ uint2 row[SEP_ROWS];
  __shared__ uint32_t kind[SEP_ROWS];
  const int64_t r = int64_t(blockIdx.x) * SEP_ROWS + threadIdx.x / SEP_QL_COUNT;
  const uint32_t lig = threadIdx.x & (SEP_QL_COUNT - 1);
  const uint32_t k = r < n ? pack[r] >> 30 : 0u;
  uint32_t ca = 0, cb = 0;
  if (k) {
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(val), 0, int(v_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t rc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(ci), 0, int(v_bytes / 2u), 0x00020000);
    const uint32_t end = uint32_t(rp[r + 1]);
    for (uint32_t e = uint32_t(rp[r]) + 4u * lig; e < end; e += 4u * SEP_QL_COUNT) {
      double w[4];
      uint32_t c[4];
      sep_values4(rv, e, w);
      sep_columns4(rc, e, c);
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t kc = (e + j < end && w[j] != 0.0) ? pack[c[j]] >> 30 : 0u;
        ca += kc == 1u;
        cb += kc == 2u;
      }
    }
  }
  ca = uint32_t(group_sum<SEP_QL_COUNT>(int(ca)));
  cb = uint32_t(group_sum<SEP_QL_COUNT>(int(cb)));
  if (lig == 0) {
    const uint2 c = make_uint2(ca, cb);
    if (r < n) counts[r] = c;
    row[threadIdx.x / SEP_QL_COUNT] = c;
    kind[threadIdx.x / SEP_QL_COUNT] = k;
  }
  __syncthreads();
  if (threadIdx.x < 64) put_sums(kind[threadIdx.x], row[threadIdx.x], int(threadIdx.x), blockIdx.x, sums, n_groups);
}

// A wave per SEP_ROWS rows.  First a lane per row: the rows' offsets from their
// counts, and their row pointers.  Where every entry of the rows goes to K_aa
// (nearly everywhere: no restrained dof near, no zero entry) the output is the
// input's run of entries with other column numbers, and the wave copies it as
// such, in 16-byte chunks aligned to the output and without regard to rows.  The
// other groups are left to sep_fill_rows (left), with their rows' first slots in
// counts.  On the 512 x 512 plate (31 M entries) 157 us for 745 MB, 4.7 TB/s, a
// large copy's rate; row by row the fill took 199 us.
__global__ __launch_bounds__(256) void sep_fill_runs(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                     const double* __restrict__ val, const uint32_t* __restrict__ pack,
                                                     uint2* __restrict__ counts, uint8_t* __restrict__ left,
                                                     const int64_t* __restrict__ off, int64_t n_groups,
                                                     const int64_t* __restrict__ head, int64_t n,
                                                     int64_t* __restrict__ out_rp, int32_t* __restrict__ out_ci,
                                                     double* __restrict__ out_v, int64_t* __restrict__ summary,
                                                     uint32_t v_bytes) {
  const int lane = threadIdx.x & 63;
  const int64_t g = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (g >= n_groups) return;
  const int64_t na = head[1], nb = head[2];
  const int64_t r0 = g * SEP_ROWS, r = r0 + lane, r1 = r0 + SEP_ROWS < n ? r0 + SEP_ROWS : n;
  const uint32_t pr = r < n ? pack[r] : 0u, k = pr >> 30;
  const uint2 c = k ? counts[r] : make_uint2(0u, 0u);
  const uint32_t first = uint32_t(rp[r0]), entries = uint32_t(rp[r1]) - first;
  // sums within 64 rows stay below 2^32: a rows' in the low half, b rows' in the high
  const uint64_t ca = k == 1u ? uint64_t(c.x) : uint64_t(c.x) << 32, cb = k == 1u ? uint64_t(c.y) : uint64_t(c.y) << 32;
  const uint64_t ia = wave_scan(ca), ib = wave_scan(cb);
  const bool run = uint32_t(__shfl(int(lo32(ia)), 63)) == entries;
  const uint32_t to = uint32_t(off[g]);  // the rows' first slot of K_aa
  if (k) {
    const int w0 = k == 1u ? 0 : 2;
    const int64_t ea = off[w0 * n_groups + g] + int64_t(k == 1u ? lo32(ia) : hi32(ia));
    const int64_t eb = off[(w0 + 1) * n_groups + g] + int64_t(k == 1u ? lo32(ib) : hi32(ib));
    // matrix w's row pointers start at start_w + w (rows_w + 1 entries, first 0)
    const int64_t pi = int64_t(pr & SEP_IDX) + 1;
    const int64_t s0 = k == 1u ? 0 : 2 * na + 2, s1 = s0 + (k == 1u ? na : nb) + 1;
    out_rp[s0 + pi] = ea - (w0 ? off[2 * n_groups] : 0);
    out_rp[s1 + pi] = eb - off[(w0 + 1) * n_groups];
    if (!run) counts[r] = make_uint2(uint32_t(ea - c.x), uint32_t(eb - c.y));
  }
  if (lane == 0) left[g] = !run;
  if (g == 0 && lane < 4) {
    const int64_t start[4] = {0, na + 1, 2 * na + 2, 2 * na + nb + 3};
    out_rp[start[lane]] = 0;
    const int64_t b = lane ? off[lane * n_groups] : 0;
    summary[3 + lane] = off[(lane + 1) * n_groups] - b;
    summary[7 + lane] = b;
    if (lane < 3) summary[lane] = head[lane];
  }
  if (!run || entries == 0) return;
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(val), 0, int(v_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(ci), 0, int(v_bytes / 2u), 0x00020000);
  const __amdgpu_buffer_rsrc_t ov = __builtin_amdgcn_make_buffer_rsrc(out_v, 0, int(v_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t oc = __builtin_amdgcn_make_buffer_rsrc(out_ci, 0, int(v_bytes / 2u), 0x00020000);
  const uint32_t end = to + entries, shift = first - to;  // input position = output position + shift (mod 2^32)
  constexpr int UV = 4, UC = 2;                           // chunks of a lane in flight
  // a chunk reaches past the run at its two ends only; what is loaded there (or
  // reads as 0 outside the array) is not stored
  for (uint32_t o = (to & ~3u) + 4u * lane; o < end; o += 4u * 64u * UC) {
    uint32_t p[UC][4];
#pragma unroll
    for (int u = 0; u < UC; ++u) sep_columns4(rc, o + 256u * u + shift, p[u]);
#pragma unroll
    for (int u = 0; u < UC; ++u) {
      const uint32_t at = o + 256u * u;
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) p[u][j] = (at + j >= to && at + j < end) ? pack[p[u][j]] & SEP_IDX : 0u;
    }
#pragma unroll
    for (int u = 0; u < UC; ++u) {
      const uint32_t at = o + 256u * u;
      if (at >= to && at + 4 <= end) {
        __builtin_amdgcn_raw_buffer_store_b128(sep_u32x4{p[u][0], p[u][1], p[u][2], p[u][3]}, oc, 4u * at, 0, 0);
      } else {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
          if (at + j >= to && at + j < end) out_ci[at + j] = int32_t(p[u][j]);
      }
    }
  }
  for (uint32_t o = (to & ~1u) + 2u * lane; o < end; o += 2u * 64u * UV) {
    sep_u32x4 x[UV];
#pragma unroll
    for (int u = 0; u < UV; ++u) x[u] = __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * (o + 128u * u + shift), 0, 0);
#pragma unroll
    for (int u = 0; u < UV; ++u) {
      const uint32_t at = o + 128u * u;
      if (at >= to && at + 2 <= end) {
        __builtin_amdgcn_raw_buffer_store_b128(x[u], ov, 8u * at, 0, 0);
      } else {
        const double2 v = __builtin_bit_cast(double2, x[u]);
        if (at >= to && at < end) out_v[at] = v.x;
        if (at + 1 >= to && at + 1 < end) out_v[at + 1] = v.y;
      }
    }
  }
}

// The groups that sep_fill_runs left, 32 rows of a group at a time.  Eight lanes
// per row, four neighbouring entries per lane and step.  Output slots in entry
// order: an exclusive scan of the per-lane counts over the row's lanes (lane l
// holds entries 4l .. 4l + 3 of the step), then each lane's entries in turn.  A
// lane whose four entries all go to an a column writes its four consecutive
// slots as two 16-byte value stores and one 16-byte column store.  A grid that
// fills the chip takes the groups in turn, 64 flags per load: a wave per eight
// rows cost 34 us where nearly none had work.
constexpr int SEP_QL_FILL = 8;
constexpr unsigned SEP_FILL_BLOCKS = 2048;
__global__ __launch_bounds__(256) void sep_fill_rows(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                     const double* __restrict__ val, const uint32_t* __restrict__ pack,
                                                     const uint2* __restrict__ counts, const uint8_t* __restrict__ left,
                                                     int64_t n_groups, int64_t n, int32_t* __restrict__ out_ci,
                                                     double* __restrict__ out_v, uint32_t v_bytes) {
  const int lane = threadIdx.x & 63;
  const uint32_t lig = lane & (SEP_QL_FILL - 1);
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(val), 0, int(v_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(ci), 0, int(v_bytes / 2u), 0x00020000);
  // outputs: the four matrices' values and columns together hold at most nnz entries
  const __amdgpu_buffer_rsrc_t ov = __builtin_amdgcn_make_buffer_rsrc(out_v, 0, int(v_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t oc = __builtin_amdgcn_make_buffer_rsrc(out_ci, 0, int(v_bytes / 2u), 0x00020000);
  for (int64_t i0 = 0; blockIdx.x + i0 * gridDim.x < n_groups; i0 += 64) {
    const int64_t mine = blockIdx.x + (i0 + lane) * gridDim.x;
    uint64_t todo = __ballot(mine < n_groups && left[mine < n_groups ? mine : 0] != 0);
    while (todo) {
      const int64_t g = blockIdx.x + (i0 + __builtin_ctzll(todo)) * gridDim.x;
      todo &= todo - 1;
#pragma unroll 1
      for (int half = 0; half < 2; ++half) {
        const int64_t r = g * SEP_ROWS + 32 * half + int(threadIdx.x) / SEP_QL_FILL;
        if (r >= n || pack[r] >> 30 == 0u) continue;    // the eight lanes of a row together
        uint32_t o_a = counts[r].x, o_b = counts[r].y;  // next slots of an a column and of a b column
        const uint32_t end = uint32_t(rp[r + 1]);
        for (uint32_t b0 = uint32_t(rp[r]); b0 < end; b0 += 4 * SEP_QL_FILL) {
          const uint32_t e = b0 + 4 * lig;
          double w[4];
          uint32_t c[4], q[4];
          sep_values4(rv, e, w);
          sep_columns4(rc, e, c);
          uint32_t la = 0, lb = 0;
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) {
            q[j] = (e + j < end && w[j] != 0.0) ? pack[c[j]] : 0u;
            la += (q[j] >> 30) == 1u;
            lb += (q[j] >> 30) == 2u;
          }
          uint32_t sum = la | lb << 16;  // at most 32 each: one scan for both
#pragma unroll
          for (uint32_t o = 1; o < SEP_QL_FILL; o <<= 1) {
            const uint32_t t = uint32_t(__shfl_up(int(sum), o, SEP_QL_FILL));
            if (lig >= o) sum += t;
          }
          const uint32_t tot = uint32_t(__shfl(int(sum), SEP_QL_FILL - 1, SEP_QL_FILL));
          uint32_t ia = o_a + (sum & 0xFFFFu) - la, ib = o_b + (sum >> 16) - lb;
          o_a += tot & 0xFFFFu;
          o_b += tot >> 16;
          if (la == 4) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(sep_u32x4, make_double2(w[0], w[1])), ov, 8u * ia, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(sep_u32x4, make_double2(w[2], w[3])), ov, 8u * ia + 16u, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(
                sep_u32x4{q[0] & SEP_IDX, q[1] & SEP_IDX, q[2] & SEP_IDX, q[3] & SEP_IDX}, oc, 4u * ia, 0, 0);
            continue;
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t kc = q[j] >> 30;
            if (kc == 1u) {
              out_ci[ia] = int32_t(q[j] & SEP_IDX);
              out_v[ia] = w[j];
              ++ia;
            } else if (kc == 2u) {
              out_ci[ib] = int32_t(q[j] & SEP_IDX);
              out_v[ib] = w[j];
              ++ib;
            }
          }
        }
      }
    }
  }
}

// Matrix w's row pointers start at out_rp[start_w + w] (rows_w + 1 entries, first 0).
__global__ void sep_finish(const uint64_t* __restrict__ pos, const int64_t* __restrict__ off,
                           const int64_t* __restrict__ err, int64_t n, int64_t* __restrict__ out_rp,
                           int64_t* __restrict__ summary) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t na = lo32(pos[n]), nb = hi32(pos[n]);
  const int64_t start[4] = {0, na, 2 * na, 2 * na + nb};
  const int64_t rows[4] = {na, na, nb, nb};
  if (t == 0) {
    summary[0] = err[0];
    summary[1] = na;
    summary[2] = nb;
    for (int w = 0; w < 4; ++w) {
      summary[3 + w] = off[start[w] + rows[w]] - off[start[w]];
      summary[7 + w] = off[start[w]];
    }
    summary[11] = 0;
  }
  if (t >= 2 * (na + nb) + 4) return;
  int w = 0;
  while (w < 3 && t >= start[w + 1] + w + 1) ++w;
  const int64_t i = t - start[w] - w;  // 0 .. rows_w
  out_rp[t] = off[start[w] + i] - off[start[w]];
}

}  // namespace

std::string upload_bc(Device* d, const uint8_t* constrained, const double* disp, const double* force, size_t n) {
  std::string e;
  if (!(e = dgrow(d->sep_cons, d->sep_cap[0], n)).empty()) return e;
  if (!(e = dgrow(d->sep_disp, d->sep_cap[1], n)).empty()) return e;
  if (!(e = dgrow(d->sep_force, d->sep_cap[2], n)).empty()) return e;
  if (n) {
    HIP_TRY(hipMemcpy(d->sep_cons, constrained, n, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(d->sep_disp, disp, n * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(d->sep_force, force, n * sizeof(double), hipMemcpyHostToDevice));
  }
  d->sep_bc_rows = int64_t(n);
  d->sep_n_cons = int64_t(n) - int64_t(std::count(constrained, constrained + n, uint8_t(0)));
  return "";
}

namespace {

// the launches of the four-entry kernels; the summary goes to sep_host
std::string separate_quad(Device* d, int64_t n, hipStream_t s, bool timed) {
  const size_t un = size_t(n);
  const unsigned chunks = unsigned((n + SEP_CHUNK - 1) / SEP_CHUNK), groups = unsigned((n + SEP_ROWS - 1) / SEP_ROWS);
  const uint32_t v_bytes = uint32_t(size_t(d->nnz) * 8);
  const int scan = int(4 * groups + 1);
  std::string e;
  if (!(e = dgrow(d->sep_pack, d->sep_cap[19], un)).empty()) return e;
  if (!(e = dgrow(d->sep_mark, d->sep_cap[20], un)).empty()) return e;
  if (!(e = dgrow(d->sep_chunk, d->sep_cap[21], size_t(chunks))).empty()) return e;
  if (!(e = dgrow(d->sep_err, d->sep_cap[22], size_t(chunks))).empty()) return e;
  if (!(e = dgrow(d->sep_rows2, d->sep_cap[23], 2 * un)).empty()) return e;
  if (!(e = dgrow(d->sep_left, d->sep_cap[24], size_t(groups))).empty()) return e;
  if (!(e = dgrow(d->sep_cnt, d->sep_cap[7], size_t(scan))).empty()) return e;
  if (!(e = dgrow(d->sep_off, d->sep_cap[8], size_t(scan))).empty()) return e;
  size_t bytes = 0;
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, d->sep_cnt, d->sep_off, scan, s));
  if (!(e = dgrow(d->sep_tmp, d->sep_cap[17], bytes)).empty()) return e;
  uint2* counts = reinterpret_cast<uint2*>(d->sep_rows2);
  if (timed) HIP_TRY(hipEventRecord(d->ev4, s));
  const unsigned waves = (groups + 3) / 4;  // workgroups of four groups
  // few restrained dofs: rows away from them are counted without their columns
  const bool few = d->sep_n_cons * SEP_FEW <= n;
  if (few)
    sep_values<<<waves, 256, 0, s>>>(d->row_ptr, d->sep_dpos, d->val, d->sep_cons, n, counts, d->sep_cls, d->sep_mark,
                                     v_bytes);
  else
    sep_diagonals<<<unsigned((n + 255) / 256), 256, 0, s>>>(d->sep_dpos, d->val, d->sep_cons, n, d->sep_cls);
  sep_classes<<<chunks, 256, 0, s>>>(d->sep_cls, d->sep_cons, n, d->sep_chunk, d->sep_err);
  sep_chunks<<<1, 1024, 0, s>>>(d->sep_chunk, d->sep_err, int(chunks), d->sep_sum);
  sep_pack_rows<<<chunks, 256, 0, s>>>(d->sep_cls, d->sep_chunk, d->sep_force, d->sep_disp, n, d->sep_pack, d->sep_aa,
                                       d->sep_bb, d->sep_ra, d->sep_ub);
  if (few) {
    sep_mark<<<waves, 256, 0, s>>>(d->row_ptr, d->col_idx, d->sep_cls, n, d->sep_mark);
    sep_count_rows<<<waves, 256, 0, s>>>(d->row_ptr, d->col_idx, d->val, d->sep_pack, d->sep_mark, n, counts,
                                         d->sep_cnt, int64_t(groups));
  } else {
    sep_count_all<<<groups, SEP_ROWS * SEP_QL_COUNT, 0, s>>>(d->row_ptr, d->col_idx, d->val, d->sep_pack, n, counts,
                                                             d->sep_cnt, int64_t(groups), v_bytes);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(d->sep_tmp, bytes, d->sep_cnt, d->sep_off, scan, s));
  sep_fill_runs<<<waves, 256, 0, s>>>(d->row_ptr, d->col_idx, d->val, d->sep_pack, counts, d->sep_left, d->sep_off,
                                      int64_t(groups), d->sep_sum, n, d->sep_rp, d->sep_ci, d->sep_v, d->sep_host,
                                      v_bytes);
  sep_fill_rows<<<few ? std::min(groups, SEP_FILL_BLOCKS) : groups, 256, 0, s>>>(d->row_ptr, d->col_idx, d->val, d->sep_pack, counts,
                                                                  d->sep_left, int64_t(groups), n, d->sep_ci, d->sep_v,
                                                                  v_bytes);
  HIP_TRY(hipGetLastError());
  return "";
}

// the launches of the one-entry kernels
std::string separate_lanes(Device* d, int64_t n, int lanes_opt, hipStream_t s, bool timed) {
  const size_t un = size_t(n);
  std::string e;
  if (!(e = dgrow(d->sep_flag, d->sep_cap[4], un + 1)).empty()) return e;
  if (!(e = dgrow(d->sep_pos, d->sep_cap[5], un + 1)).empty()) return e;
  if (!(e = dgrow(d->sep_key, d->sep_cap[6], un)).empty()) return e;
  if (!(e = dgrow(d->sep_cnt, d->sep_cap[7], 2 * un + 1)).empty()) return e;
  if (!(e = dgrow(d->sep_off, d->sep_cap[8], 2 * un + 1)).empty()) return e;
  // scratch of the hipCUB reduction and scans: the largest of the three
  size_t b0 = 0, b1 = 0, b2 = 0;
  HIP_TRY(hipcub::DeviceReduce::Min(nullptr, b0, d->sep_key, d->sep_sum + SEP_SUMMARY, int(n), s));
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, b1, d->sep_flag, d->sep_pos, int(n + 1), s));
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, b2, d->sep_cnt, d->sep_off, int(2 * n + 1), s));
  if (!(e = dgrow(d->sep_tmp, d->sep_cap[17], std::max(b0, std::max(b1, b2)))).empty()) return e;
  const unsigned B = 256;
  // lanes per row: the option's, else 8 (4 for rows shorter than 8 entries on average)
  const int lanes = lanes_opt ? lanes_opt : (d->nnz / n >= 8 ? 8 : 4);
  const unsigned G = unsigned((n * lanes + B - 1) / B);
  auto count = lanes == 32 ? sep_count<32> : lanes == 16 ? sep_count<16> : lanes == 8 ? sep_count<8> : sep_count<4>;
  auto fill = lanes == 32 ? sep_fill<32> : lanes == 16 ? sep_fill<16> : lanes == 8 ? sep_fill<8> : sep_fill<4>;
  if (timed) HIP_TRY(hipEventRecord(d->ev4, s));
  sep_classify<<<unsigned((n + 1 + B - 1) / B), B, 0, s>>>(d->sep_dpos, d->val, d->sep_cons, n, d->sep_cls,
                                                           d->sep_flag, d->sep_key, d->sep_cnt);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipcub::DeviceReduce::Min(d->sep_tmp, b0, d->sep_key, d->sep_sum + SEP_SUMMARY, int(n), s));
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(d->sep_tmp, b1, d->sep_flag, d->sep_pos, int(n + 1), s));
  count<<<G, B, 0, s>>>(d->row_ptr, d->col_idx, d->val, d->sep_cls, d->sep_pos, d->sep_force, d->sep_disp, n,
                        d->sep_cnt, d->sep_aa, d->sep_bb, d->sep_ra, d->sep_ub);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(d->sep_tmp, b2, d->sep_cnt, d->sep_off, int(2 * n + 1), s));
  fill<<<G, B, 0, s>>>(d->row_ptr, d->col_idx, d->val, d->sep_cls, d->sep_pos, d->sep_off, n, d->sep_ci, d->sep_v);
  HIP_TRY(hipGetLastError());
  sep_finish<<<unsigned((2 * n + 4 + B - 1) / B), B, 0, s>>>(d->sep_pos, d->sep_off, d->sep_sum + SEP_SUMMARY, n,
                                                            d->sep_rp, d->sep_host);
  HIP_TRY(hipGetLastError());
  return "";
}

}  // namespace

std::string separate_sparse(Device* d, SepResult& res, void* stream, bool timed, int lanes_opt) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t n = d->n_rows;
  res = SepResult();
  d->sep_done = false;
  d->sep_ms = 0.0;
  if (n >= int64_t(INT32_MAX) / 2) return "too many rows for the separation";
  if (lanes_opt != 0 && lanes_opt != 4 && lanes_opt != 8 && lanes_opt != 16 && lanes_opt != 32)
    return "lanes per row must be 0 (automatic), 4, 8, 16 or 32";
  if (d->sep_bc_rows != n) return "boundary conditions are not uploaded";
  if (n == 0) return "";  // no dof: no restraints
  const size_t un = size_t(n);
  // four entries per lane (sep_*_quad) while the values span under 4 GiB; an
  // explicit lanes option (or larger values) takes the one-entry kernels
  const bool quad = lanes_opt == 0 && size_t(d->nnz) * 8 < (size_t(1) << 32);
  std::string e;
  if (!(e = dgrow(d->sep_cls, d->sep_cap[3], un)).empty()) return e;
  if (!(e = dgrow(d->sep_aa, d->sep_cap[9], un)).empty()) return e;
  if (!(e = dgrow(d->sep_bb, d->sep_cap[10], un)).empty()) return e;
  if (!(e = dgrow(d->sep_ra, d->sep_cap[11], un)).empty()) return e;
  if (!(e = dgrow(d->sep_ub, d->sep_cap[12], un)).empty()) return e;
  if (!(e = dgrow(d->sep_rp, d->sep_cap[13], 2 * un + 4)).empty()) return e;
  if (!(e = dgrow(d->sep_ci, d->sep_cap[14], size_t(d->nnz))).empty()) return e;
  if (!(e = dgrow(d->sep_v, d->sep_cap[15], size_t(d->nnz))).empty()) return e;
  if (!(e = dgrow(d->sep_sum, d->sep_cap[16], size_t(SEP_SUMMARY + 1))).empty()) return e;
  if (!d->sep_host) HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&d->sep_host), SEP_SUMMARY * sizeof(int64_t)));
  const unsigned B = 256;
  if (!d->sep_dpos_valid) {
    if (!(e = dgrow(d->sep_dpos, d->sep_cap[18], un)).empty()) return e;
    sep_diag_pos<<<unsigned((n + B - 1) / B), B, 0, s>>>(d->row_ptr, d->col_idx, n, d->sep_dpos);
    HIP_TRY(hipGetLastError());
    d->sep_dpos_valid = true;
  }
  e = quad ? separate_quad(d, n, s, timed) : separate_lanes(d, n, lanes_opt, s, timed);
  if (!e.empty()) return e;
  if (timed) HIP_TRY(hipEventRecord(d->ev5, s));
  HIP_TRY(hipStreamSynchronize(s));
  const int64_t* sum = d->sep_host;
  res.err_row = sum[0] == INT64_MAX ? -1 : sum[0];
  res.n_aa = sum[1];
  res.n_bb = sum[2];
  for (int w = 0; w < 4; ++w) {
    res.nnz[w] = sum[3 + w];
    d->sep_base[w] = sum[7 + w];
  }
  d->sep_rows[0] = d->sep_rows[1] = res.n_aa;
  d->sep_rows[2] = d->sep_rows[3] = res.n_bb;
  for (int w = 0; w < 4; ++w) d->sep_nnz[w] = res.nnz[w];
  d->sep_done = true;
  if (timed) {
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, d->ev4, d->ev5));
    d->sep_ms = ms;
  }
  return "";
}

std::string separated_csr(Device* d, int which, const int64_t** rp, const int32_t** ci, const double** v) {
  if (which < 0 || which > 3 || !d->sep_done) return "no separation computed";
  const int64_t start[4] = {0, d->sep_rows[0], 2 * d->sep_rows[0], 2 * d->sep_rows[0] + d->sep_rows[2]};
  if (rp) *rp = d->sep_rp + start[which] + which;
  if (ci) *ci = d->sep_ci + d->sep_base[which];
  if (v) *v = d->sep_v + d->sep_base[which];
  return "";
}

std::string separated_vectors(Device* d, const int64_t** aa, const int64_t** bb, const double** r_a,
                              const double** u_b) {
  if (!d->sep_done) return "no separation computed";
  if (aa) *aa = d->sep_aa;
  if (bb) *bb = d->sep_bb;
  if (r_a) *r_a = d->sep_ra;
  if (u_b) *u_b = d->sep_ub;
  return "";
}

void separation_shape(Device* d, int64_t rows[4], int64_t nnz[4]) {
  for (int w = 0; w < 4; ++w) {
    if (rows) rows[w] = d->sep_done ? d->sep_rows[w] : 0;
    if (nnz) nnz[w] = d->sep_done ? d->sep_nnz[w] : 0;
  }
}

void invalidate_separation(Device* d) { d->sep_done = false; }

double last_separate_ms(Device* d) { return d->sep_ms; }

}  // namespace femdev
