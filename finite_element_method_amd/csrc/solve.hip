// solve.hip -- the crate's sparse global analysis on the device
// (methods_for_global_analysis.rs:28-133, 135-275):
//   b   = r_a - K_ab u_b                                  (find_b_sparse)
//   K_aa u_a = b by preconditioned conjugate gradients, Jacobi or node-block
//   Jacobi                       (pcg_jacobi_csr / pcg_block_jacobi_csr)
//   r_r = (K_ba u_a + K_bb u_b) - r_b                     (find_r_r_sparse)
// on the matrices of the last separation (separate.hip).
//
// PCG is Saad's Algorithm 9.1 with x0 = 0, stopped when
// ||r||_2 <= max(rel_tol ||b||_2, abs_tol) and counting the x updates.  All
// reductions use a grid that depends on n only and fixed trees, so a solve is
// bitwise reproducible.  The scalars (alpha, beta, r.z) stay on the device.
//
// An update is four launches: product, p.Ap, the vector update and the
// direction.  The last two begin by summing the partial sums of the one before
// in every workgroup (the same tree, so every workgroup has the same bits),
// which takes the place of two one-workgroup launches per update.  Up to FU_N
// rows it is two (sv_direction_product).
//
// Small systems (SM_N rows, SM_NNZ entries) are solved by one workgroup, sv_small.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>

#include "device_state.hpp"
#include "fem_device.hpp"
#include "lane_ops.hpp"

namespace femdev {

namespace {

constexpr int SV_B = 256;         // threads per block of the vector kernels
constexpr int SV_PARTS = 1024;    // most blocks of the reductions
constexpr int SPMV_LANES = 8;     // lanes per CSR row
constexpr int BJ_MAX = 6;         // dofs per node block

// scalar slots (device).  r.z and the stop flag (converged or capped: every
// later kernel of the loop returns at once) have two slots: update u reads slot
// u & 1 and its last kernel writes the other, so that no workgroup reads what
// another of the same launch writes.
enum { S_RZ = 0, S_DONE = 2, S_RR = 4, S_BB, S_STATUS, S_ITER, S_CONV, S_COUNT };
constexpr int BJ_PER_WAVE = 10;   // node blocks per wave in the block-Jacobi kernels (6 lanes each)

template <class T>
std::string dgrow(T*& p, size_t& cap, size_t n) {
  if (n <= cap && p) return "";
  auto e = dalloc(p, n ? n : 1);
  if (!e.empty()) { cap = 0; return e; }
  cap = n ? n : 1;
  return "";
}

// y[r] = (base ? base[r] : 0) + sign * (A x)[r] - (sub ? sub[r] : 0); SPMV_LANES lanes per row,
// each summing its strided entries in order, combined by a fixed butterfly.
__global__ void sv_spmv(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci, const double* __restrict__ v,
                        const double* __restrict__ x, const double* base, double sign, const double* __restrict__ sub,
                        double* y, int64_t n) {
  const int64_t r = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / SPMV_LANES;
  const int lig = threadIdx.x & (SPMV_LANES - 1);
  if (r >= n) return;
  double acc = 0.0;
  for (int64_t e = rp[r] + lig; e < rp[r + 1]; e += SPMV_LANES) acc += v[e] * x[ci[e]];
#pragma unroll
  for (int o = SPMV_LANES / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, SPMV_LANES);
  if (lig == 0) {
    double out = base ? base[r] + sign * acc : sign * acc;
    if (sub) out -= sub[r];
    y[r] = out;
  }
}

// Ap = K p inside the update loop (returns at once after the stop flag).
// SPMV_QUAD_LANES lanes per row, each taking four neighbouring values per step
// with two 16-byte value loads and one 16-byte column load, range-checked
// buffer loads (32-bit offsets: below 4 GiB of values).  On the plate matrices
// (rows of 9 to 27 values) this beats one 8-byte load per lane and value by
// about a fifth: fewer, fuller memory requests.  Fixed summation order (each
// lane's values in turn, then a butterfly over the row's lanes).
constexpr int SPMV_QUAD_LANES = 4;
__global__ void sv_spmv_it_quad(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                const double* __restrict__ v, const double* __restrict__ p, double* __restrict__ ap,
                                int64_t n, const double* s, int turn, uint32_t v_bytes) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  if (s[S_DONE + turn] != 0.0) return;
  const int64_t r = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / SPMV_QUAD_LANES;
  const int lig = threadIdx.x & (SPMV_QUAD_LANES - 1);
  if (r >= n) return;
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(v), 0, int(v_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(ci), 0, int(v_bytes / 2u), 0x00020000);
  const int64_t end = rp[r + 1];
  double acc = 0.0;
  for (int64_t e = rp[r] + 4 * lig; e < end; e += 4 * SPMV_QUAD_LANES) {
    const uint32_t ev = uint32_t(e);
    // values and columns past the row end (or the array end: read as 0) are
    // loaded but not used; their columns are valid indices or 0
    const double2 w0 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * ev, 0, 0));
    const double2 w1 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * ev + 16u, 0, 0));
    const u32x4 c = __builtin_amdgcn_raw_buffer_load_b128(rc, 4u * ev, 0, 0);
    acc = __builtin_fma(w0.x, p[int32_t(c.x)], acc);
    if (e + 1 < end) acc = __builtin_fma(w0.y, p[int32_t(c.y)], acc);
    if (e + 2 < end) acc = __builtin_fma(w1.x, p[int32_t(c.z)], acc);
    if (e + 3 < end) acc = __builtin_fma(w1.y, p[int32_t(c.w)], acc);
  }
#pragma unroll
  for (int o = SPMV_QUAD_LANES / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, SPMV_QUAD_LANES);
  if (lig == 0) ap[r] = acc;
}

// the same with one 8-byte load per lane and value (values beyond 4 GiB)
__global__ void sv_spmv_it(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                           const double* __restrict__ v, const double* __restrict__ p, double* __restrict__ ap,
                           int64_t n, const double* s, int turn) {
  if (s[S_DONE + turn] != 0.0) return;
  const int64_t r = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / SPMV_LANES;
  const int lig = threadIdx.x & (SPMV_LANES - 1);
  if (r >= n) return;
  double acc = 0.0;
  for (int64_t e = rp[r] + lig; e < rp[r + 1]; e += SPMV_LANES) acc = __builtin_fma(v[e], p[ci[e]], acc);
#pragma unroll
  for (int o = SPMV_LANES / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, SPMV_LANES);
  if (lig == 0) ap[r] = acc;
}

// ---- K_aa in slices, for the update loop
//
// The CSR product above moves 12 bytes per entry and spends its memory
// instructions on rows of 9 to 27 entries split over four lanes.  A solve that
// goes on after its first update copies K_aa once into slices of 64 rows, a lane
// per row:
//   * every value load of a wave is 1 KiB of consecutive bytes;
//   * a column takes 16 bits from the slice's lowest column while the slice spans
//     under 2^16 columns, 32 bits otherwise;
//   * rows are sorted by length within windows of SL_WINDOW rows, so that the
//     lanes of a slice end together (a plate's rows of 18, 27 and 1 entries
//     alternate).
// A row's entries go to four partial sums, combined as sv_spmv_it_quad's four
// lanes combine theirs, entry for entry: the product has the same bits, and the
// rows' order in the slices does not show.
//
// Slice s, at its offset of 256-byte units: `pairs` x 64 value pairs (16 bytes a
// lane), then `pairs` x 64 column pairs (4 bytes a lane, or 8).
//
// Bound: the entries' stream, 10.3 bytes per entry with the padding; on the
// 512 x 512 plate (31 M entries) 78 us per product, 4.1 TB/s, against 106 us for
// the CSR product; without the gathers of p it would take 62-68 us.  Measured and
// left out: rows with equal columns sharing a lane (fewer columns and gathers,
// but each gather then spans 64 nodes: 188 us), one 16-byte gather for two
// neighbouring columns (87 us), an XCD-contiguous order of the slices (no change).
constexpr int SL_WINDOW = 1024;  // rows sorted together, by one workgroup
// The copy costs about two CSR products and a fixed 50 us.  From 10 M entries
// on a solve of 20 updates gains it back (17 M entries: 2.04 vs 2.11 ms, 50
// updates 4.47 vs 4.88; 7.7 M entries: 1.22 vs 1.16 ms, 50 updates 2.66 vs 2.64).
constexpr int64_t SL_MIN_NNZ = 10000000;    // K_aa entries
constexpr int SL_MIN_UPDATES = 16;          // updates asked for
// Bytes per entry up to which the slices are taken.  A slice is as wide as its
// longest row: a few long rows per window (hubs) cost all 64 lanes their length.
// 10.3 bytes take 78 us where the CSR product takes 106, so the gain ends at
// 14; a lattice with a hub of 400 bars among every 341 nodes would take some 50 bytes,
// in time and in memory that the handle then keeps.
constexpr size_t SL_MAX_BYTES = 14;
constexpr uint32_t SL_NONE = 0xFFFFFFFFu;   // no row in this lane
constexpr uint32_t SL_UNITS16 = 5, SL_UNITS32 = 6;  // 256-byte units of a pair of 64 lanes

__device__ inline uint32_t wave_min(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, uint32_t(__shfl_xor(int(v), o)));
  return v;
}
__device__ inline uint32_t wave_max(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, uint32_t(__shfl_xor(int(v), o)));
  return v;
}

// one workgroup per window: rows in order of (length, index); per slice its
// pairs | wide << 31, lowest column and size in units.  Lengths are below 2^22
// (the pattern's rows are bounded by 65535 plus a block).
__global__ __launch_bounds__(512) void sv_slice_rows(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                     int64_t n, uint32_t* __restrict__ rows,
                                                     uint32_t* __restrict__ pairs, uint32_t* __restrict__ cbase,
                                                     uint32_t* __restrict__ units, int64_t n_slices) {
  __shared__ uint32_t key[SL_WINDOW];
  const int64_t w0 = int64_t(blockIdx.x) * SL_WINDOW;
  for (int i = threadIdx.x; i < SL_WINDOW; i += 512) {
    const int64_t r = w0 + i;
    key[i] = r < n ? uint32_t(rp[r + 1] - rp[r]) << 10 | uint32_t(i) : SL_NONE;
  }
  __syncthreads();
  for (int k = 2; k <= SL_WINDOW; k <<= 1)  // bitonic sort, ascending
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < SL_WINDOW / 2; t += 512) {
        const int i = 2 * t - (t & (j - 1)), o = i + j;
        const uint32_t a = key[i], b = key[o];
        if ((a > b) == ((i & k) == 0)) {
          key[i] = b;
          key[o] = a;
        }
      }
      __syncthreads();
    }
  const int lane = threadIdx.x & 63;
  for (int q = threadIdx.x >> 6; q < SL_WINDOW / 64; q += 8) {
    const int64_t s = int64_t(blockIdx.x) * (SL_WINDOW / 64) + q;
    const uint32_t kk = key[64 * q + lane];
    const bool on = kk != SL_NONE;
    const int64_t r = w0 + int64_t(kk & (SL_WINDOW - 1));
    const uint32_t len = on ? kk >> 10 : 0u;
    uint32_t lo = SL_NONE, hi = 0u;
    if (len) {  // columns ascend within a row
      const int64_t b = rp[r];
      lo = uint32_t(ci[b]);
      hi = uint32_t(ci[b + len - 1]);
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    const uint32_t np = (wave_max(len) + 1u) >> 1;
    if (s >= n_slices) continue;
    rows[64 * s + lane] = on ? uint32_t(r) : SL_NONE;
    if (lane == 0) {
      const bool wide = np && hi - lo > 0xFFFFu;
      pairs[s] = np | uint32_t(wide) << 31;
      cbase[s] = np ? lo : 0u;
      units[s] = np * (wide ? SL_UNITS32 : SL_UNITS16);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) units[n_slices] = 0u;  // totals slot of the scan
}

// One wave per slice.  16 entries of each of 64 rows at a time go through LDS:
// four lanes read a row's 16 entries together (range-checked 16-byte loads: what
// lies past a row or the array is loaded but not kept), then each lane writes
// the pairs of its own row, so that reads and writes both cover consecutive
// bytes.  Unused places hold value 0 and the slice's lowest column.
constexpr int SL_TILE = 17;
__device__ inline void sl_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__global__ __launch_bounds__(256) void sv_slice_fill(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                     const double* __restrict__ v, const uint32_t* __restrict__ rows,
                                                     const uint32_t* __restrict__ pairs,
                                                     const uint32_t* __restrict__ cbase,
                                                     const uint32_t* __restrict__ offset, int64_t n_slices,
                                                     unsigned char* __restrict__ data, uint32_t v_bytes) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  __shared__ double tile_v[4][64 * SL_TILE];
  __shared__ uint32_t tile_c[4][64 * SL_TILE];
  const int64_t s = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (s >= n_slices) return;
  const uint32_t pw = pairs[s], np = pw & 0x7FFFFFFFu, cb = cbase[s], r = rows[64 * s + lane];
  const bool wide = pw >> 31;
  double* tv = tile_v[threadIdx.x >> 6];
  uint32_t* tc = tile_c[threadIdx.x >> 6];
  const uint32_t first = r == SL_NONE ? 0u : uint32_t(rp[r]);  // positions are below 2^29
  const uint32_t len = r == SL_NONE ? 0u : uint32_t(rp[r + 1]) - first;
  double2* dv = reinterpret_cast<double2*>(data + size_t(offset[s]) * 256);
  uint32_t* dc = reinterpret_cast<uint32_t*>(dv + 64 * size_t(np));
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(v), 0, int(v_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(ci), 0, int(v_bytes / 2u), 0x00020000);
  for (uint32_t j0 = 0; j0 < np; j0 += 8) {
    double2 x0[4], x1[4];
    u32x4 cc[4];
    uint32_t left[4];  // entries of the row from the lane's first on
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {  // 16 rows, one per four lanes
      const int src = 16 * pass + (lane >> 2);
      const uint32_t sl = uint32_t(__shfl(int(len), src)), e = 2 * j0 + 4 * (lane & 3);
      const uint32_t at = uint32_t(__shfl(int(first), src)) + e;
      left[pass] = e < sl ? sl - e : 0u;
      x0[pass] = x1[pass] = make_double2(0.0, 0.0);
      cc[pass] = u32x4{0u, 0u, 0u, 0u};
      if (left[pass]) {
        x0[pass] = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * at, 0, 0));
        x1[pass] = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * at + 16u, 0, 0));
        cc[pass] = __builtin_amdgcn_raw_buffer_load_b128(rc, 4u * at, 0, 0);
      }
    }
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
      const int o = SL_TILE * (16 * pass + (lane >> 2)) + 4 * (lane & 3);
      const uint32_t n = left[pass];
      tv[o] = n > 0 ? x0[pass].x : 0.0;
      tv[o + 1] = n > 1 ? x0[pass].y : 0.0;
      tv[o + 2] = n > 2 ? x1[pass].x : 0.0;
      tv[o + 3] = n > 3 ? x1[pass].y : 0.0;
      tc[o] = n > 0 ? cc[pass].x - cb : 0u;
      tc[o + 1] = n > 1 ? cc[pass].y - cb : 0u;
      tc[o + 2] = n > 2 ? cc[pass].z - cb : 0u;
      tc[o + 3] = n > 3 ? cc[pass].w - cb : 0u;
    }
    sl_lds_sync();
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j)
      if (j0 + j < np) {
        const double* t = tv + SL_TILE * lane + 2 * j;
        const uint32_t c0 = tc[SL_TILE * lane + 2 * j], c1 = tc[SL_TILE * lane + 2 * j + 1];
        dv[64 * size_t(j0 + j) + lane] = make_double2(t[0], t[1]);
        if (wide)
          reinterpret_cast<uint2*>(dc)[64 * size_t(j0 + j) + lane] = make_uint2(c0, c1);
        else
          dc[64 * size_t(j0 + j) + lane] = c0 | c1 << 16;
      }
    sl_lds_sync();
  }
}

// N column pairs from pair j: all loads first, then pairs 0, 1 into partial sum
// a and 2, 3 into b.  The entries are read once per product: non-temporal, so
// that p keeps the caches (88 -> 78 us on the 512 x 512 plate).  Places past a
// row's end are loaded (value 0) but not summed, so that an infinite or NaN
// entry of p reaches only the rows that hold its column.
template <bool WIDE, int N>
__device__ inline void slice_pairs(const double2* __restrict__ dv, const uint32_t* __restrict__ dc,
                                   const double* __restrict__ p, uint32_t j, uint32_t len, int lane, double& a,
                                   double& b) {
  typedef double sl_d2 __attribute__((ext_vector_type(2)));
  typedef unsigned int sl_u2 __attribute__((ext_vector_type(2)));
  sl_d2 w[N];
  sl_d2 x[N];
#pragma unroll
  for (int t = 0; t < N; ++t) {
    uint32_t c0, c1;
    if (WIDE) {
      const sl_u2 c = __builtin_nontemporal_load(reinterpret_cast<const sl_u2*>(dc) + 64 * size_t(j + t) + lane);
      c0 = c.x;
      c1 = c.y;
    } else {
      const uint32_t c = __builtin_nontemporal_load(dc + 64 * size_t(j + t) + lane);
      c0 = c & 0xFFFFu;
      c1 = c >> 16;
    }
    w[t] = __builtin_nontemporal_load(reinterpret_cast<const sl_d2*>(dv) + 64 * size_t(j + t) + lane);
    x[t].x = p[c0];
    x[t].y = p[c1];
  }
#pragma unroll
  for (int t = 0; t < N; ++t) {
    double& acc = t < 2 ? a : b;
    if (2 * (j + t) < len) acc = __builtin_fma(w[t].x, x[t].x, acc);
    if (2 * (j + t) + 1 < len) acc = __builtin_fma(w[t].y, x[t].y, acc);
  }
}

template <bool WIDE>
__device__ inline double slice_row(const double2* __restrict__ dv, const uint32_t* __restrict__ dc,
                                   const double* __restrict__ p, uint32_t np, uint32_t len, int lane) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  uint32_t j = 0;
  // four pairs (two quads of columns) into two partial sums; false after the
  // last ones.  np is the slice's, so the whole wave takes the same way.
  auto chunk = [&](double& a, double& b) -> bool {
    const uint32_t left = np - j;
    if (left < 4) {
      if (left == 1) slice_pairs<WIDE, 1>(dv, dc, p, j, len, lane, a, b);
      if (left == 2) slice_pairs<WIDE, 2>(dv, dc, p, j, len, lane, a, b);
      if (left == 3) slice_pairs<WIDE, 3>(dv, dc, p, j, len, lane, a, b);
      return false;
    }
    slice_pairs<WIDE, 4>(dv, dc, p, j, len, lane, a, b);
    j += 4;
    return true;
  };
  while (chunk(a0, a1) && chunk(a2, a3)) {
  }
  return (a0 + a2) + (a1 + a3);
}

__global__ __launch_bounds__(256) void sv_spmv_slices(const unsigned char* __restrict__ data,
                                                      const int64_t* __restrict__ rp,
                                                      const uint32_t* __restrict__ rows,
                                                      const uint32_t* __restrict__ pairs,
                                                      const uint32_t* __restrict__ cbase,
                                                      const uint32_t* __restrict__ offset, int64_t n_slices,
                                                      const double* __restrict__ p, double* __restrict__ ap,
                                                      const double* s, int turn) {
  if (s[S_DONE + turn] != 0.0) return;
  const int64_t sl = int64_t(__builtin_amdgcn_readfirstlane(int(blockIdx.x * 4 + (threadIdx.x >> 6))));
  const int lane = threadIdx.x & 63;
  if (sl >= n_slices) return;
  const uint32_t pw = pairs[sl], np = pw & 0x7FFFFFFFu, r = rows[64 * sl + lane];
  const double2* dv = reinterpret_cast<const double2*>(data + size_t(offset[sl]) * 256);
  const uint32_t* dc = reinterpret_cast<const uint32_t*>(dv + 64 * size_t(np));
  const uint32_t len = r == SL_NONE ? 0u : uint32_t(rp[r + 1] - rp[r]);
  const double* q = p + cbase[sl];
  const double y = pw >> 31 ? slice_row<true>(dv, dc, q, np, len, lane) : slice_row<false>(dv, dc, q, np, len, lane);
  if (r != SL_NONE) ap[r] = y;
}

// sums of two values over the block, in every thread: a butterfly per wave,
// then the waves in order
struct Sum2 {
  double a, b;
};
__device__ inline Sum2 block_sum2(double a, double b) {
  __shared__ Sum2 w[SV_B / 64];
  a = wave_sum(a);
  b = wave_sum(b);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = {a, b};
  __syncthreads();
  Sum2 t = w[0];
#pragma unroll
  for (int k = 1; k < SV_B / 64; ++k) {
    t.a += w[k].a;
    t.b += w[k].b;
  }
  __syncthreads();  // w may be written again
  return t;
}

// the block's sums into its partials (part_b may be absent)
__device__ inline void block_partials(double a, double b, double* part_a, double* part_b) {
  const Sum2 t = block_sum2(a, b);
  if (threadIdx.x == 0) {
    part_a[blockIdx.x] = t.a;
    if (part_b) part_b[blockIdx.x] = t.b;
  }
}

// total of the partials of a launch of the same grid, in every thread
__device__ inline Sum2 total_partials(const double* part_a, const double* part_b) {
  double a = 0.0, b = 0.0;
  for (unsigned i = threadIdx.x; i < gridDim.x; i += SV_B) {
    a += part_a[i];
    if (part_b) b += part_b[i];
  }
  return block_sum2(a, b);
}

// partials of p.Ap
__global__ __launch_bounds__(SV_B) void sv_dot_it(const double* __restrict__ x, const double* __restrict__ y, int64_t n,
                                                  const double* s, int turn, double* part) {
  if (s[S_DONE + turn] != 0.0) return;
  double a = 0.0;
  for (int64_t i = int64_t(blockIdx.x) * SV_B + threadIdx.x; i < n; i += int64_t(gridDim.x) * SV_B)
    a = __builtin_fma(x[i], y[i], a);
  block_partials(a, 0.0, part, nullptr);
}

// start: r.z and b.b from the partials of the start kernel (one workgroup)
__global__ __launch_bounds__(SV_B) void sv_start_scalars(const double* __restrict__ part_a,
                                                         const double* __restrict__ part_b, int parts, double* s) {
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < parts; i += SV_B) {
    a += part_a[i];
    b += part_b[i];
  }
  const Sum2 t = block_sum2(a, b);
  if (threadIdx.x == 0) {
    s[S_RZ] = t.a;
    s[S_BB] = t.b;
    s[S_RR] = t.b;
  }
}

// Jacobi: d[i] = K_aa(i, i)
__global__ void sv_diag(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci, const double* __restrict__ v,
                        int64_t n, double* __restrict__ d) {
  const int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r >= n) return;
  double dd = 0.0;
  for (int64_t e = rp[r]; e < rp[r + 1]; ++e)
    if (ci[e] == r) dd = v[e];
  d[r] = dd;
}

// node blocks of K_aa: flag[i] = row i starts a node (methods_for_global_analysis.rs:135-160)
__global__ void sv_block_flags(const int64_t* __restrict__ aa, int64_t n, uint32_t* __restrict__ flag) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i > n) return;
  flag[i] = i < n && (i == 0 || aa[i] / 6 != aa[i - 1] / 6);
}
__global__ void sv_block_starts(const uint32_t* __restrict__ flag, const uint32_t* __restrict__ id, int64_t n,
                                int32_t* __restrict__ starts) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i > n) return;
  if (i == n) starts[id[n]] = int32_t(n);  // id[n] = number of blocks
  else if (flag[i]) starts[id[i]] = int32_t(i);
}

// inverse of each node block (Gauss-Jordan, partial pivoting); status bit 1 on a
// singular block.  `count`, where given, holds the number of blocks (nblk is then its bound).
__global__ __launch_bounds__(256) void sv_block_inverse(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                        const double* __restrict__ v,
                                                        const int32_t* __restrict__ starts, int64_t nblk,
                                                        const uint32_t* __restrict__ count,
                                                        double* __restrict__ inv, double* s) {
  // The augmented block [A | I] lives in registers: every loop below runs over
  // compile-time indices, so row swaps and column placement are selects (a
  // runtime-indexed array would sit in scratch memory).  A block of m < 6 dofs
  // is padded with the identity: its rows and columns past m never become
  // pivots or elimination targets of the first m columns, so the m x m inverse
  // is the one the unpadded elimination gives.
  const int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (b >= (count ? int64_t(*count) : nblk)) return;
  const int s0 = starts[b], m = starts[b + 1] - s0;
  double* o = inv + 36 * b;
  if (m > BJ_MAX) {  // a node has at most six dofs; guard the fixed-size arrays anyway
    for (int i = 0; i < 36; ++i) o[i] = 0.0;
    s[S_STATUS] = 1.0;
    return;
  }
  double a[BJ_MAX][2 * BJ_MAX];
#pragma unroll
  for (int i = 0; i < BJ_MAX; ++i) {
#pragma unroll
    for (int j = 0; j < 2 * BJ_MAX; ++j) a[i][j] = (j == BJ_MAX + i || (i >= m && j == i)) ? 1.0 : 0.0;
    if (i < m) {
      // the block's columns s0 .. s0 + m - 1 are one run of the sorted row:
      // find its start by bisection, then place at most m entries
      int64_t lo = rp[s0 + i], hi = rp[s0 + i + 1];
      const int64_t end = hi;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (ci[mid] < s0) lo = mid + 1; else hi = mid;
      }
      for (int64_t e = lo; e < end; ++e) {
        const int c = ci[e] - s0;
        if (c >= m) break;
        const double x = v[e];
#pragma unroll
        for (int j = 0; j < BJ_MAX; ++j) a[i][j] = c == j ? x : a[i][j];
      }
    }
  }
  bool ok = true;
#pragma unroll
  for (int c = 0; c < BJ_MAX; ++c) {
    // partial pivoting: the first row of largest |a[i][c]|, i >= c
    int piv = c;
    double best = fabs(a[c][c]);
#pragma unroll
    for (int i = c + 1; i < BJ_MAX; ++i)
      if (fabs(a[i][c]) > best) {
        piv = i;
        best = fabs(a[i][c]);
      }
    ok = ok && best != 0.0;
#pragma unroll
    for (int i = c + 1; i < BJ_MAX; ++i) {
      const bool sw = piv == i;
#pragma unroll
      for (int j = 0; j < 2 * BJ_MAX; ++j) {
        const double t = a[c][j];
        a[c][j] = sw ? a[i][j] : t;
        a[i][j] = sw ? t : a[i][j];
      }
    }
    const double d = a[c][c];
#pragma unroll
    for (int j = 0; j < 2 * BJ_MAX; ++j) a[c][j] /= d;
#pragma unroll
    for (int i = 0; i < BJ_MAX; ++i)
      if (i != c) {
        const double f = a[i][c];
#pragma unroll
        for (int j = 0; j < 2 * BJ_MAX; ++j) a[i][j] = f != 0.0 ? a[i][j] - f * a[c][j] : a[i][j];
      }
  }
#pragma unroll
  for (int i = 0; i < BJ_MAX; ++i)
#pragma unroll
    for (int j = 0; j < BJ_MAX; ++j) o[6 * i + j] = (i < m && j < m) ? a[i][BJ_MAX + j] : 0.0;
  if (!ok) s[S_STATUS] = 1.0;  // any writer stores the same value
}

// start: r = b, z = M^-1 r, p = z, partials of (r, z) and (b, b)
__global__ void sv_start_jacobi(const double* __restrict__ b, const double* __restrict__ d, int64_t n,
                                double* __restrict__ x, double* __restrict__ r, double* __restrict__ z,
                                double* __restrict__ p, double* part_a, double* part_b) {
  double ra = 0.0, rb = 0.0;
  for (int64_t i = int64_t(blockIdx.x) * SV_B + threadIdx.x; i < n; i += int64_t(gridDim.x) * SV_B) {
    const double bi = b[i], zi = bi / d[i];
    x[i] = 0.0;
    r[i] = bi;
    z[i] = zi;
    p[i] = zi;
    ra = __builtin_fma(bi, zi, ra);
    rb = __builtin_fma(bi, bi, rb);
  }
  block_partials(ra, rb, part_a, part_b);
}

// update: x += alpha p, r -= alpha Ap, z = r / d; partials of (r, z) and (r, r)
__global__ void sv_update_jacobi(const double* __restrict__ d, const double* __restrict__ p,
                                 const double* __restrict__ ap, const double* __restrict__ s, int turn,
                                 const double* __restrict__ part_pap, int64_t n, double* __restrict__ x,
                                 double* __restrict__ r, double* __restrict__ z, double* part_a, double* part_b) {
  if (s[S_DONE + turn] != 0.0) return;
  const double alpha = s[S_RZ + turn] / total_partials(part_pap, nullptr).a;
  double ra = 0.0, rb = 0.0;
  for (int64_t i = int64_t(blockIdx.x) * SV_B + threadIdx.x; i < n; i += int64_t(gridDim.x) * SV_B) {
    x[i] = __builtin_fma(alpha, p[i], x[i]);
    const double ri = __builtin_fma(-alpha, ap[i], r[i]);
    r[i] = ri;
    const double zi = ri / d[i];
    z[i] = zi;
    ra = __builtin_fma(ri, zi, ra);
    rb = __builtin_fma(ri, ri, rb);
  }
  block_partials(ra, rb, part_a, part_b);
}

// block Jacobi: six lanes per node block (lane = row of the block), ten
// blocks per wave; z = M^-1 r with the row of the inverse read as three
// 16-byte loads and the block's r gathered by lane shuffles.  Lanes beyond
// a block's size, and the last four lanes of each wave, only take part in the
// shuffles.
struct BjLane {
  int64_t k;  // node block
  int row, s0, m;
  bool act;   // row < m of an existing block
};
__device__ inline BjLane bj_lane(const int32_t* __restrict__ starts, int64_t nblk, int64_t wave, int lane) {
  BjLane o;
  o.k = wave * BJ_PER_WAVE + lane / 6;
  o.row = lane % 6;
  o.s0 = 0;
  o.m = 0;
  if (lane < 6 * BJ_PER_WAVE && o.k < nblk) {
    o.s0 = starts[o.k];
    o.m = starts[o.k + 1] - o.s0;
  }
  o.act = o.row < o.m;
  return o;
}
__device__ inline void bj_row(const double* __restrict__ inv, const BjLane& L, double w[6]) {
  double2 w0 = make_double2(0.0, 0.0), w1 = w0, w2 = w0;
  if (L.act) {
    const double2* row = reinterpret_cast<const double2*>(inv + 36 * L.k + 6 * L.row);
    w0 = row[0];
    w1 = row[1];
    w2 = row[2];
  }
  w[0] = w0.x; w[1] = w0.y; w[2] = w1.x; w[3] = w1.y; w[4] = w2.x; w[5] = w2.y;
}
__device__ inline double bj_apply(const double w[6], const BjLane& L, int lane, double ri) {
  double zi = 0.0;
  const int first = lane - L.row;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const double rj = __shfl(ri, (first + j) & 63);  // every lane takes part
    if (j < L.m) zi = __builtin_fma(w[j], rj, zi);
  }
  return zi;
}
__device__ inline double bj_row_apply(const double* __restrict__ inv, const BjLane& L, int lane, double ri) {
  double w[6];
  bj_row(inv, L, w);
  return bj_apply(w, L, lane, ri);
}
__global__ void sv_start_block(const double* __restrict__ b, const double* __restrict__ inv,
                               const int32_t* __restrict__ starts, int64_t nblk, double* __restrict__ x,
                               double* __restrict__ r, double* __restrict__ z, double* __restrict__ p, double* part_a,
                               double* part_b) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = int64_t(gridDim.x) * (SV_B / 64);
  double ra = 0.0, rb = 0.0;
  for (int64_t w = int64_t(blockIdx.x) * (SV_B / 64) + (threadIdx.x >> 6); w * BJ_PER_WAVE < nblk; w += waves) {
    const BjLane L = bj_lane(starts, nblk, w, lane);
    double ri = 0.0;
    if (L.act) {
      const int64_t i = L.s0 + L.row;
      ri = b[i];
      x[i] = 0.0;
      r[i] = ri;
    }
    const double zi = bj_row_apply(inv, L, lane, ri);
    if (L.act) {
      const int64_t i = L.s0 + L.row;
      z[i] = zi;
      p[i] = zi;
      ra = __builtin_fma(ri, zi, ra);
      rb = __builtin_fma(ri, ri, rb);
    }
  }
  block_partials(ra, rb, part_a, part_b);
}
// update: x += alpha p, r -= alpha Ap, z = M^-1 r; partials of (r, z) and (r, r)
__global__ void sv_update_block(const double* __restrict__ inv, const int32_t* __restrict__ starts, int64_t nblk,
                                const double* __restrict__ p, const double* __restrict__ ap,
                                const double* __restrict__ s, int turn, const double* __restrict__ part_pap,
                                double* __restrict__ x, double* __restrict__ r, double* __restrict__ z, double* part_a,
                                double* part_b) {
  if (s[S_DONE + turn] != 0.0) return;
  const double alpha = s[S_RZ + turn] / total_partials(part_pap, nullptr).a;
  const int lane = threadIdx.x & 63;
  const int64_t waves = int64_t(gridDim.x) * (SV_B / 64);
  double ra = 0.0, rb = 0.0;
  for (int64_t w = int64_t(blockIdx.x) * (SV_B / 64) + (threadIdx.x >> 6); w * BJ_PER_WAVE < nblk; w += waves) {
    const BjLane L = bj_lane(starts, nblk, w, lane);
    double ri = 0.0;
    if (L.act) {
      const int64_t i = L.s0 + L.row;
      x[i] = __builtin_fma(alpha, p[i], x[i]);
      ri = __builtin_fma(-alpha, ap[i], r[i]);
      r[i] = ri;
    }
    const double zi = bj_row_apply(inv, L, lane, ri);
    if (L.act) {
      z[L.s0 + L.row] = zi;
      ra = __builtin_fma(ri, zi, ra);
      rb = __builtin_fma(ri, ri, rb);
    }
  }
  block_partials(ra, rb, part_a, part_b);
}

// beta and the update's scalars from the partials of (r, z) and (r, r); p = z + beta p
__global__ __launch_bounds__(SV_B) void sv_direction(const double* __restrict__ z, double* s, int turn,
                                                     const double* __restrict__ part_a,
                                                     const double* __restrict__ part_b, double stop, double max_iter,
                                                     int64_t n, double* __restrict__ p) {
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (s[S_DONE + turn] != 0.0) {
    if (first) s[S_DONE + (turn ^ 1)] = 1.0;  // the flag goes on to the next update
    return;
  }
  const Sum2 t = total_partials(part_a, part_b);
  const double beta = t.a / s[S_RZ + turn];
  if (first) {
    s[S_RZ + (turn ^ 1)] = t.a;
    s[S_RR] = t.b;
    const double it = s[S_ITER] + 1.0;
    const bool conv = sqrt(t.b) <= stop;
    s[S_ITER] = it;
    s[S_CONV] = conv ? 1.0 : 0.0;
    s[S_DONE + (turn ^ 1)] = (conv || it >= max_iter) ? 1.0 : 0.0;
  }
  for (int64_t i = int64_t(blockIdx.x) * SV_B + threadIdx.x; i < n; i += int64_t(gridDim.x) * SV_B)
    p[i] = __builtin_fma(beta, p[i], z[i]);
}

// ---- small systems: the whole solve in one workgroup
//
// Up to SM_N rows the update loop above is launches and the gaps between them
// (four per update, a host wait per batch), its work a few hundred KiB.  Here
// one workgroup keeps the vectors in LDS and runs the updates behind barriers.
// Bound: K_aa read from L2 by one CU (64 B per clock) and the chain of its
// product, two sums and the preconditioner.  Sums follow the grid kernels' trees
// (a "virtual wave" here is a wave of theirs), so both ways have the same bits.
// 50 block-Jacobi updates with their set-up, grid kernels and here:
//   rows 24 (24 updates) 657 -> 99 us; 192: 895 -> 226; 1008 (18 k entries):
//   900 -> 383; 1649 (30 k): 961 -> 547; 1275 (62 k): 979 -> 731; 1649 (82 k):
//   973 -> 845.
// SM_NNZ is where that ends: one CU's reading of 100 k entries costs an update
// of the grid kernels.  SM_N is the size of the vectors in LDS (91 KB).
constexpr int SM_T = 1024;
constexpr int64_t SM_N = 2048;
constexpr int64_t SM_NNZ = 80 * 1024;
constexpr int SM_CHUNK = 4096;               // updates per launch, so that no launch runs on unboundedly
constexpr int SM_VW = int(SM_N) / 64;        // virtual waves

// zeroes the scalars; for node blocks their starts and number (one workgroup)
__global__ __launch_bounds__(SM_T) void sv_small_setup(const int64_t* __restrict__ aa, int n, bool blocks,
                                                       int32_t* __restrict__ starts, uint32_t* __restrict__ count,
                                                       double* __restrict__ s) {
  __shared__ uint32_t waves[SM_T / 64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (t < S_COUNT) s[t] = 0.0;
  if (!blocks) return;
  uint32_t before = 0;
  for (int base = 0; base < n; base += SM_T) {
    const int i = base + t;
    const bool flag = i < n && (i == 0 || aa[i] / 6 != aa[i - 1] / 6);
    const uint64_t m = __ballot(flag);
    if (lane == 0) waves[wave] = uint32_t(__popcll(m));
    __syncthreads();
    uint32_t at = before + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
    for (int w = 0; w < SM_T / 64; ++w) {
      if (w < wave) at += waves[w];
      before += waves[w];
    }
    if (flag) starts[at] = i;
    __syncthreads();
  }
  if (t == 0) {
    starts[before] = n;
    *count = before;
  }
}

// sums of a virtual wave's two values into slot vw
__device__ inline void small_wave_sum(double a, double b, int vw, Sum2* slots) {
  a = wave_sum(a);
  b = wave_sum(b);
  if ((threadIdx.x & 63) == 0) slots[vw] = {a, b};
}
// total_partials of `parts` blocks (at most eight) of four virtual waves, in
// every thread: the steps of the butterfly that would add zeros are left out
__device__ inline Sum2 small_total(const Sum2* slots, int parts) {
  const int lane = threadIdx.x & 7;
  Sum2 t{0.0, 0.0};
  if (lane < parts) {
    t = slots[4 * lane];
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      t.a += slots[4 * lane + k].a;
      t.b += slots[4 * lane + k].b;
    }
  }
  t.a += lane_xor<4>(t.a);
  t.b += lane_xor<4>(t.b);
  t.a += lane_xor<2>(t.a);
  t.b += lane_xor<2>(t.b);
  t.a += lane_xor<1>(t.a);
  t.b += lane_xor<1>(t.b);
  return t;
}

// four neighbouring entries of K_aa (zeros past the end of the array)
struct SmQuad {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  double2 w0, w1;
  u32x4 c;
};
__device__ inline SmQuad small_quad(__amdgpu_buffer_rsrc_t rv, __amdgpu_buffer_rsrc_t rc, uint32_t e) {
  SmQuad q;
  q.w0 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * e, 0, 0));
  q.w1 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * e + 16u, 0, 0));
  q.c = __builtin_amdgcn_raw_buffer_load_b128(rc, 4u * e, 0, 0);
  return q;
}

template <bool BLOCK>
__global__ __launch_bounds__(SM_T) void sv_small(const int64_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                 const double* __restrict__ v, uint32_t v_bytes,
                                                 const double* __restrict__ b, const double* __restrict__ diag,
                                                 const double* __restrict__ inv, const int32_t* __restrict__ starts,
                                                 const uint32_t* __restrict__ count, int n, int parts, double rel_tol,
                                                 double abs_tol, int max_iter, bool resume, double* __restrict__ x,
                                                 double* __restrict__ r, double* __restrict__ p, double* s) {
  __shared__ double lx[SM_N], lr[SM_N], lz[SM_N], lp[SM_N], lap[SM_N];
  __shared__ uint32_t lrp[SM_N + 1];
  __shared__ Sum2 dots[SM_VW], sums[SM_VW];
  if (BLOCK && s[S_STATUS] != 0.0) return;  // a singular block: the host reports it
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nvw = 4 * parts;
  const int64_t nblk = BLOCK ? int64_t(*count) : 0;
  // the preconditioner of the wave's first two turns, kept: rows of the block
  // inverses (turns w = wave and w1), or diagonal entries (virtual waves wave, wave + 16)
  const int w1 = wave + (nvw <= SM_T / 64 ? nvw : SM_T / 64);
  BjLane k0{}, k1{};
  double inv0[6], inv1[6], d0 = 1.0, d1 = 1.0;
  if (BLOCK) {
    k0 = bj_lane(starts, nblk, wave, lane);
    k1 = bj_lane(starts, nblk, w1, lane);
    bj_row(inv, k0, inv0);
    bj_row(inv, k1, inv1);
  } else {
    if (t < n) d0 = diag[t];
    if (t + SM_T < n) d1 = diag[t + SM_T];
  }
  for (int i = t; i <= n; i += SM_T) lrp[i] = uint32_t(rp[i]);
  double rz, rr, bb;
  int it = 0;
  if (resume) {
    for (int i = t; i < n; i += SM_T) {
      lx[i] = x[i];
      lr[i] = r[i];
      lp[i] = p[i];
    }
    rz = s[S_RZ];
    rr = s[S_RR];
    bb = s[S_BB];
    it = int(s[S_ITER]);
    __syncthreads();  // thread 0 writes the scalars at the end
  } else {
    for (int vw = wave; vw < nvw; vw += SM_T / 64) {
      double ra = 0.0, rb = 0.0;
      if (BLOCK) {
        for (int64_t w = vw; w * BJ_PER_WAVE < nblk; w += nvw) {
          const BjLane L = bj_lane(starts, nblk, w, lane);
          const int i = L.s0 + L.row;
          const double ri = L.act ? b[i] : 0.0;
          const double zi = bj_row_apply(inv, L, lane, ri);
          if (L.act) {
            lx[i] = 0.0;
            lr[i] = ri;
            lp[i] = zi;
            ra = __builtin_fma(ri, zi, ra);
            rb = __builtin_fma(ri, ri, rb);
          }
        }
      } else if (64 * vw + lane < n) {
        const int i = 64 * vw + lane;
        const double bi = b[i], zi = bi / (vw == wave ? d0 : d1);
        lx[i] = 0.0;
        lr[i] = bi;
        lp[i] = zi;
        ra = __builtin_fma(bi, zi, 0.0);
        rb = __builtin_fma(bi, bi, 0.0);
      }
      small_wave_sum(ra, rb, vw, sums);
    }
    __syncthreads();
    const Sum2 t2 = small_total(sums, parts);
    rz = t2.a;
    rr = t2.b;
    bb = t2.b;
  }
  const double rel = rel_tol * sqrt(bb);
  const double stop = rel < abs_tol ? abs_tol : rel;
  bool conv = sqrt(rr) <= stop;
  bool done = conv || it >= max_iter;
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(v), 0, int(v_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(ci), 0, int(v_bytes / 2u), 0x00020000);
  // every thread has the same scalars, so all leave the loop together
#pragma unroll 1
  for (int k = 0; k < SM_CHUNK && !done; ++k) {
    __syncthreads();
    // Ap = K p: sv_spmv_it_quad's four lanes per row, two rows per lane, each
    // row's next entries loaded while the last ones are summed
    const int lig = t & 3;
    for (int r0 = t >> 2; r0 < n; r0 += 2 * (SM_T / 4)) {
      const int r1 = r0 + SM_T / 4;
      uint32_t e[2] = {lrp[r0] + 4u * lig, 0u}, end[2] = {lrp[r0 + 1], 0u};
      if (r1 < n) {
        e[1] = lrp[r1] + 4u * lig;
        end[1] = lrp[r1 + 1];
      }
      double acc[2] = {0.0, 0.0};
      SmQuad cur[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) cur[h] = small_quad(rv, rc, e[h]);
      while (e[0] < end[0] || e[1] < end[1]) {
        SmQuad next[2];
        const bool more = e[0] + 16u < end[0] || e[1] + 16u < end[1];
        if (more) {
#pragma unroll
          for (int h = 0; h < 2; ++h) next[h] = small_quad(rv, rc, e[h] + 16u);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // past a row's end: loaded, not summed
          const double p0 = lp[cur[h].c.x], p1 = lp[cur[h].c.y], p2 = lp[cur[h].c.z], p3 = lp[cur[h].c.w];
          if (e[h] < end[h]) acc[h] = __builtin_fma(cur[h].w0.x, p0, acc[h]);
          if (e[h] + 1 < end[h]) acc[h] = __builtin_fma(cur[h].w0.y, p1, acc[h]);
          if (e[h] + 2 < end[h]) acc[h] = __builtin_fma(cur[h].w1.x, p2, acc[h]);
          if (e[h] + 3 < end[h]) acc[h] = __builtin_fma(cur[h].w1.y, p3, acc[h]);
          e[h] += 16u;
        }
        if (!more) break;
#pragma unroll
        for (int h = 0; h < 2; ++h) cur[h] = next[h];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        acc[h] += lane_xor<2>(acc[h]);
        acc[h] += lane_xor<1>(acc[h]);
      }
      if (lig == 0) {
        lap[r0] = acc[0];
        if (r1 < n) lap[r1] = acc[1];
      }
    }
    __syncthreads();
    for (int vw = wave; vw < nvw; vw += SM_T / 64) {
      const int i = 64 * vw + lane;
      small_wave_sum(i < n ? __builtin_fma(lp[i], lap[i], 0.0) : 0.0, 0.0, vw, dots);
    }
    __syncthreads();
    const double alpha = rz / small_total(dots, parts).a;
    for (int vw = wave; vw < nvw; vw += SM_T / 64) {
      double ra = 0.0, rb = 0.0;
      if (BLOCK) {
        for (int w = vw; w * BJ_PER_WAVE < nblk; w += nvw) {
          BjLane L = w == wave ? k0 : k1;
          double row[6];
#pragma unroll
          for (int j = 0; j < 6; ++j) row[j] = w == wave ? inv0[j] : inv1[j];
          if (w != wave && w != w1) {
            L = bj_lane(starts, nblk, w, lane);
            bj_row(inv, L, row);
          }
          const int i = L.s0 + L.row;
          double ri = 0.0;
          if (L.act) {
            lx[i] = __builtin_fma(alpha, lp[i], lx[i]);
            ri = __builtin_fma(-alpha, lap[i], lr[i]);
            lr[i] = ri;
          }
          const double zi = bj_apply(row, L, lane, ri);
          if (L.act) {
            lz[i] = zi;
            ra = __builtin_fma(ri, zi, ra);
            rb = __builtin_fma(ri, ri, rb);
          }
        }
      } else if (64 * vw + lane < n) {
        const int i = 64 * vw + lane;
        lx[i] = __builtin_fma(alpha, lp[i], lx[i]);
        const double ri = __builtin_fma(-alpha, lap[i], lr[i]);
        lr[i] = ri;
        const double zi = ri / (vw == wave ? d0 : d1);
        lz[i] = zi;
        ra = __builtin_fma(ri, zi, 0.0);
        rb = __builtin_fma(ri, ri, 0.0);
      }
      small_wave_sum(ra, rb, vw, sums);
    }
    __syncthreads();
    const Sum2 t2 = small_total(sums, parts);
    const double beta = t2.a / rz;
    rz = t2.a;
    rr = t2.b;
    ++it;
    conv = sqrt(rr) <= stop;
    done = conv || it >= max_iter;
    for (int i = t; i < n; i += SM_T) lp[i] = __builtin_fma(beta, lp[i], lz[i]);
  }
  __syncthreads();
  for (int i = t; i < n; i += SM_T) {
    x[i] = lx[i];
    r[i] = lr[i];
    p[i] = lp[i];
  }
  if (t == 0) {
    s[S_RZ] = rz;
    s[S_RR] = rr;
    s[S_BB] = bb;
    s[S_ITER] = double(it);
    s[S_CONV] = conv ? 1.0 : 0.0;
    s[S_DONE] = done ? 1.0 : 0.0;
  }
}

// ---- two launches per update
//
// For systems of up to FU_N rows an update of four launches is mostly launches.
// Here the direction, K p and p.Ap are one: a workgroup owns 256 rows, forms the
// entries of p that its columns name from the last z and p (the same fused
// multiply-add that sv_direction does, so the same bits in every workgroup),
// writes its own to `p_new` and its partial of p.Ap.  The other launch is the
// vector update.  Sums follow the trees of sv_dot_it and sv_direction: the same
// bits.  50 block-Jacobi updates with set-up, four launches and two:
//   plates of 2541 rows 1001 -> 770 us, 14161: 969 -> 805, 55969: 1021 -> 866;
//   frame of 45600: 1020 -> 850; trusses of 50700: 1053 -> 910.
// FU_N is a workgroup per CU: with 76049 rows 1131 -> 1101, 136051: 1501 -> 1517
// (a second round of workgroups, and the second gather).
// turn: the update's; its predecessor left r.z and the stop flag in turn ^ 1.
// with_direction: false for the first update after the scalars were read, whose
// p is already the direction (and stays where it is).
constexpr int64_t FU_N = 256 * SV_B;
constexpr int FU_T = 1024;
static_assert(3 * ((FU_N + SV_B - 1) / SV_B) <= 2 * SV_PARTS, "three sets of partials in the array of two");
__global__ __launch_bounds__(FU_T) void sv_direction_product(const int64_t* __restrict__ rp,
                                                             const int32_t* __restrict__ ci,
                                                             const double* __restrict__ v, uint32_t v_bytes,
                                                             const double* __restrict__ z, const double* __restrict__ p,
                                                             double* __restrict__ p_new, double* __restrict__ ap,
                                                             int64_t n, double* s, int turn, bool with_direction,
                                                             const double* __restrict__ part_a,
                                                             const double* __restrict__ part_b, double stop,
                                                             double* __restrict__ part_pap) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  __shared__ double own_p[SV_B], own_ap[SV_B];
  __shared__ Sum2 w[SV_B / 64];
  const int t = threadIdx.x;
  const bool first = blockIdx.x == 0 && t == 0;
  double beta = 0.0;
  if (!with_direction) {
    if (s[S_DONE + turn] != 0.0) return;
  } else {
    if (s[S_DONE + (turn ^ 1)] != 0.0) {
      if (first) s[S_DONE + turn] = 1.0;
      return;
    }
    const double rz = s[S_RZ + (turn ^ 1)];
    if (t < SV_B) {  // total_partials
      double a = 0.0, b = 0.0;
      for (unsigned i = t; i < gridDim.x; i += SV_B) {
        a += part_a[i];
        b += part_b[i];
      }
      a = wave_sum(a);
      b = wave_sum(b);
      if ((t & 63) == 0) w[t >> 6] = {a, b};
    }
    __syncthreads();
    Sum2 sum = w[0];
#pragma unroll
    for (int k = 1; k < SV_B / 64; ++k) {
      sum.a += w[k].a;
      sum.b += w[k].b;
    }
    __syncthreads();  // w is written again below
    beta = sum.a / rz;
    // the host queues no update past the last one, so only convergence stops here
    const bool conv = sqrt(sum.b) <= stop;
    if (first) {
      s[S_RZ + turn] = sum.a;
      s[S_RR] = sum.b;
      s[S_ITER] += 1.0;
      s[S_CONV] = conv ? 1.0 : 0.0;
      s[S_DONE + turn] = conv ? 1.0 : 0.0;
    }
    if (conv) return;
  }
  auto direction = [&](int32_t c) { return with_direction ? __builtin_fma(beta, p[c], z[c]) : p[c]; };
  // Ap = K p: sv_spmv_it_quad
  const int64_t r = int64_t(blockIdx.x) * SV_B + (t >> 2);
  const int lig = t & 3;
  if (r < n) {
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(v), 0, int(v_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t rc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(ci), 0, int(v_bytes / 2u), 0x00020000);
    const int64_t end = rp[r + 1];
    double acc = 0.0;
    for (int64_t e = rp[r] + 4 * lig; e < end; e += 4 * SPMV_QUAD_LANES) {
      const uint32_t ev = uint32_t(e);
      const double2 w0 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * ev, 0, 0));
      const double2 w1 = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(rv, 8u * ev + 16u, 0, 0));
      const u32x4 c = __builtin_amdgcn_raw_buffer_load_b128(rc, 4u * ev, 0, 0);
      // columns past the row end are valid indices or 0
      const double p0 = direction(int32_t(c.x)), p1 = direction(int32_t(c.y));
      const double p2 = direction(int32_t(c.z)), p3 = direction(int32_t(c.w));
      acc = __builtin_fma(w0.x, p0, acc);
      if (e + 1 < end) acc = __builtin_fma(w0.y, p1, acc);
      if (e + 2 < end) acc = __builtin_fma(w1.x, p2, acc);
      if (e + 3 < end) acc = __builtin_fma(w1.y, p3, acc);
    }
    acc += lane_xor<2>(acc);
    acc += lane_xor<1>(acc);
    if (lig == 0) own_ap[t >> 2] = acc;
    if (lig == 1) own_p[t >> 2] = direction(int32_t(r));
  }
  __syncthreads();
  if (t < SV_B) {
    const int64_t i = int64_t(blockIdx.x) * SV_B + t;
    double a = 0.0;
    if (i < n) {
      a = __builtin_fma(own_p[t], own_ap[t], 0.0);
      ap[i] = own_ap[t];
      if (with_direction) p_new[i] = own_p[t];
    }
    a = wave_sum(a);
    if ((t & 63) == 0) w[t >> 6] = {a, 0.0};
  }
  __syncthreads();
  if (t == 0) part_pap[blockIdx.x] = ((w[0].a + w[1].a) + w[2].a) + w[3].a;
}

// r_b: forces at the k_bb indexes
__global__ void sv_gather(const double* __restrict__ src, const int64_t* __restrict__ idx, int64_t n,
                          double* __restrict__ dst) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}

unsigned grid_for(int64_t items, int per_block) { return unsigned(std::max<int64_t>(1, (items + per_block - 1) / per_block)); }

}  // namespace

// Work buffers of one solve.  get(slot, bytes) returns device memory for a
// slot; vectors: 0 b, 1 x = u_a, 2 r, 3 z, 4 p, 5 Ap, 6 r_r, 7 r_b; 8 the
// reduction partials, 9 the scalars, 10 the Jacobi diagonal, 11 block flags,
// 12 block ids, 13 block starts, 14 scan storage, 15 block inverses; where
// grows(), also K_aa's slices: 16 rows, 17 pairs, 18 lowest columns, 19 sizes,
// 20 offsets, 21 entries.
struct SolveBuffers {
  virtual std::string get(int slot, size_t bytes, void** out) = 0;
  virtual bool grows() const { return false; }
  virtual size_t room() const { return size_t(1) << 62; }  // bytes that get() can still hand out
  double* host = nullptr;  // S_COUNT + 1 doubles of host memory for the scalar reads
};

namespace {

__global__ void sv_zero(double* __restrict__ x, int n) {
  if (int(threadIdx.x) < n) x[threadIdx.x] = 0.0;
}

template <class T>
std::string take(SolveBuffers& bufs, int slot, size_t n, T*& out) {
  void* p = nullptr;
  auto e = bufs.get(slot, std::max<size_t>(n, 1) * sizeof(T), &p);
  out = static_cast<T*>(p);
  return e;
}

// K_aa's slices (sv_spmv_slices): rows and sizes first, the entries once the
// total size has been read
struct Slices {
  int64_t n = 0;
  uint32_t *rows = nullptr, *pairs = nullptr, *cbase = nullptr, *units = nullptr, *offset = nullptr;
  unsigned char* data = nullptr;
};

std::string slices_size(SolveBuffers& bufs, const int64_t* rp, const int32_t* ci, int64_t na, hipStream_t s,
                        Slices& sl) {
  sl.n = (na + 63) / 64;
  const size_t un = size_t(sl.n);
  std::string e;
  if (!(e = take(bufs, 16, 64 * un, sl.rows)).empty()) return e;
  if (!(e = take(bufs, 17, un, sl.pairs)).empty()) return e;
  if (!(e = take(bufs, 18, un, sl.cbase)).empty()) return e;
  if (!(e = take(bufs, 19, un + 1, sl.units)).empty()) return e;
  if (!(e = take(bufs, 20, un + 1, sl.offset)).empty()) return e;
  size_t bytes = 0;
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, sl.units, sl.offset, int(un + 1), s));
  void* tmp = nullptr;
  if (!(e = bufs.get(14, std::max<size_t>(bytes, 1), &tmp)).empty()) return e;
  sv_slice_rows<<<grid_for(na, SL_WINDOW), 512, 0, s>>>(rp, ci, na, sl.rows, sl.pairs, sl.cbase, sl.units, sl.n);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, sl.units, sl.offset, int(un + 1), s));
  return "";
}

// false (and no error left behind) when there is no memory for the entries
bool slices_fill(SolveBuffers& bufs, const int64_t* rp, const int32_t* ci, const double* v, uint32_t v_bytes,
                 uint32_t units, hipStream_t s, Slices& sl) {
  void* data = nullptr;
  if (!bufs.get(21, size_t(units) * 256, &data).empty() || !data) {
    (void)hipGetLastError();
    return false;
  }
  sl.data = static_cast<unsigned char*>(data);
  sv_slice_fill<<<grid_for(sl.n, 4), 256, 0, s>>>(rp, ci, v, sl.rows, sl.pairs, sl.cbase, sl.offset, sl.n, sl.data,
                                                      v_bytes);
  return hipGetLastError() == hipSuccess;
}

// the solve proper: b, preconditioner, PCG updates, r_r, into `bufs`
std::string solve_core(Device* d, int precond, int max_iter, double rel_tol, double abs_tol, hipStream_t s,
                       SolveResult& res, bool wide, bool plain, SolveBuffers& bufs) {
  res = SolveResult();
  const int64_t na = d->sep_rows[0], nb = d->sep_rows[2];
  const size_t una = size_t(std::max<int64_t>(na, 1)), unb = size_t(std::max<int64_t>(nb, 1));
  std::string e;
  double* vec[8];
  for (int k = 0; k < 6; ++k)  // b, x, r, z, p, Ap
    if (!(e = take(bufs, k, una, vec[k])).empty()) return e;
  if (!(e = take(bufs, 6, unb, vec[6])).empty()) return e;
  if (!(e = take(bufs, 7, unb, vec[7])).empty()) return e;
  double *part = nullptr, *sc = nullptr;
  if (!(e = take(bufs, 8, size_t(2 * SV_PARTS), part)).empty()) return e;
  if (!(e = take(bufs, 9, size_t(S_COUNT), sc)).empty()) return e;
  double *b = vec[0], *x = vec[1], *r = vec[2], *z = vec[3], *p = vec[4], *ap = vec[5], *rr = vec[6], *rb = vec[7];
  double* host = bufs.host;
  const int64_t* rp[4];
  const int32_t* ci[4];
  const double* v[4];
  for (int w = 0; w < 4; ++w)
    if (!(e = separated_csr(d, w, &rp[w], &ci[w], &v[w])).empty()) return e;
  const int64_t *aa_idx = d->sep_aa, *bb_idx = d->sep_bb;
  const double *r_a = d->sep_ra, *u_b = d->sep_ub;
  const unsigned B = SV_B;
  HIP_TRY(hipEventRecord(d->ev4, s));
  // b = r_a - K_ab u_b
  if (na) {
    sv_spmv<<<grid_for(na * SPMV_LANES, B), B, 0, s>>>(rp[1], ci[1], v[1], u_b, r_a, -1.0, nullptr, b, na);
    HIP_TRY(hipGetLastError());
  }
  // preconditioner
  int64_t nblk = 0;
  double* diag = nullptr;
  double* inv = nullptr;
  int32_t* starts = nullptr;
  // the reductions' grid: one block per SV_B dofs, at most SV_PARTS (a function
  // of n, and the same for every launch of the solve)
  const unsigned parts = unsigned(std::min<int64_t>(SV_PARTS, grid_for(na, SV_B)));
  const bool quad = wide && size_t(d->sep_nnz[0]) * 8 < (size_t(1) << 32);
  const uint32_t v_bytes = quad ? uint32_t(size_t(d->sep_nnz[0]) * 8) : 0u;
  // partials: (r, z), (r, r) and p.Ap.  b is not read after the start (it holds n
  // values, at least one per block): it takes the third set, or with two launches
  // per update, whose three sets fit `part`, the other direction
  const bool fused = quad && !plain && na <= FU_N;
  constexpr int FU_PARTS = 2 * SV_PARTS / 3;
  double *pa = part, *pb = part + (fused ? FU_PARTS : SV_PARTS), *pc = fused ? part + 2 * FU_PARTS : b;
  double stop = 0.0;
  int it = 0;
  bool conv = false;
  // a small system: one block inverse per dof is room enough, so the number of
  // node blocks stays on the device, and so do the tolerance and the updates
  if (quad && !plain && na > 0 && na <= SM_N && d->sep_nnz[0] <= SM_NNZ &&
      bufs.room() >= una * (36 * sizeof(double) + sizeof(int32_t)) + 4096) {
    uint32_t* count = nullptr;
    if (precond == 0) {
      if (!(e = take(bufs, 10, una, diag)).empty()) return e;
      sv_diag<<<grid_for(na, B), B, 0, s>>>(rp[0], ci[0], v[0], na, diag);
    } else {
      if (!(e = take(bufs, 15, 36 * una, inv)).empty()) return e;
      if (!(e = take(bufs, 13, una + 1, starts)).empty()) return e;
      if (!(e = take(bufs, 12, 1, count)).empty()) return e;
    }
    sv_small_setup<<<1, SM_T, 0, s>>>(aa_idx, int(na), precond != 0, starts, count, sc);
    if (precond != 0)
      sv_block_inverse<<<grid_for(na, B), B, 0, s>>>(rp[0], ci[0], v[0], starts, na, count, inv, sc);
    auto kernel = precond == 0 ? sv_small<false> : sv_small<true>;
    bool resume = false;
    do {
      kernel<<<1, SM_T, 0, s>>>(rp[0], ci[0], v[0], v_bytes, b, diag, inv, starts, count, int(na), int(parts), rel_tol,
                                abs_tol, max_iter, resume, x, r, p, sc);
      HIP_TRY(hipGetLastError());
      HIP_TRY(hipMemcpyAsync(host, sc, sizeof(double) * S_COUNT, hipMemcpyDeviceToHost, s));
      HIP_TRY(hipStreamSynchronize(s));
      if (host[S_STATUS] != 0.0) return "PCG(BlockJacobi): singular node block";
      resume = true;
    } while (host[S_DONE] == 0.0);
    stop = std::max(rel_tol * std::sqrt(host[S_BB]), abs_tol);
    it = int(host[S_ITER]);
    conv = host[S_CONV] != 0.0;
  } else {
    sv_zero<<<1, 64, 0, s>>>(sc, S_COUNT);
    HIP_TRY(hipGetLastError());
    if (precond == 0) {
      if (!(e = take(bufs, 10, una, diag)).empty()) return e;
      if (na) {
        sv_diag<<<grid_for(na, B), B, 0, s>>>(rp[0], ci[0], v[0], na, diag);
        HIP_TRY(hipGetLastError());
      }
    } else {
      uint32_t *flag = nullptr, *bid = nullptr;
      if (!(e = take(bufs, 11, una + 1, flag)).empty()) return e;
      if (!(e = take(bufs, 12, una + 1, bid)).empty()) return e;
      if (!(e = take(bufs, 13, una + 1, starts)).empty()) return e;
      sv_block_flags<<<grid_for(na + 1, B), B, 0, s>>>(aa_idx, na, flag);
      HIP_TRY(hipGetLastError());
      size_t bytes = 0;
      HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, flag, bid, int(na + 1), s));
      void* tmp = nullptr;
      if (!(e = bufs.get(14, std::max<size_t>(bytes, 1), &tmp)).empty()) return e;
      HIP_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, flag, bid, int(na + 1), s));
      sv_block_starts<<<grid_for(na + 1, B), B, 0, s>>>(flag, bid, na, starts);
      HIP_TRY(hipGetLastError());
      uint32_t nb32 = 0;
      HIP_TRY(hipMemcpyAsync(host, bid + na, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
      HIP_TRY(hipStreamSynchronize(s));
      std::memcpy(&nb32, host, sizeof(uint32_t));
      nblk = int64_t(nb32);
      if (!(e = take(bufs, 15, size_t(36 * std::max<int64_t>(nblk, 1)), inv)).empty()) return e;
      if (nblk) {
        sv_block_inverse<<<grid_for(nblk, B), B, 0, s>>>(rp[0], ci[0], v[0], starts, nblk, nullptr, inv, sc);
        HIP_TRY(hipGetLastError());
      }
    }
    // start
    if (precond == 0)
      sv_start_jacobi<<<parts, B, 0, s>>>(b, diag, na, x, r, z, p, pa, pb);
    else
      sv_start_block<<<parts, B, 0, s>>>(b, inv, starts, nblk, x, r, z, p, pa, pb);
    HIP_TRY(hipGetLastError());
    sv_start_scalars<<<1, B, 0, s>>>(pa, pb, int(parts), sc);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(host, sc, sizeof(double) * S_COUNT, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    if (host[S_STATUS] != 0.0) return "PCG(BlockJacobi): singular node block";
    stop = std::max(rel_tol * std::sqrt(host[S_BB]), abs_tol);
    it = 0;
    conv = std::sqrt(host[S_RR]) <= stop;
    if (!conv && max_iter > 0) {
      // Updates are queued in growing batches; the last scalar kernel of an
      // update raises the stop flag on convergence or at max_iter, and every
      // kernel queued after that returns at once.  The count stays exact and the
      // host waits once per batch, not once per update.
      const unsigned spmv_blocks = grid_for(na * (quad ? SPMV_QUAD_LANES : SPMV_LANES), B);
      double* p_other = b;
      Slices sl;
      bool slice = quad && !plain && !fused && bufs.grows() && d->sep_nnz[0] >= SL_MIN_NNZ && max_iter >= SL_MIN_UPDATES;
      uint32_t slice_total = 0;
      int queued = 0, batch = 1;
      for (;;) {
        const int nq = std::min(batch, max_iter - queued);
        for (int q = 0; q < nq; ++q) {
          const int turn = (queued + q) & 1;
          if (fused) {
            sv_direction_product<<<parts, FU_T, 0, s>>>(rp[0], ci[0], v[0], v_bytes, z, p, p_other, ap, na, sc, turn,
                                                        q > 0, pa, pb, stop, pc);
            if (q > 0) std::swap(p, p_other);
          } else if (sl.data)
            sv_spmv_slices<<<grid_for(sl.n, 4), 256, 0, s>>>(sl.data, rp[0], sl.rows, sl.pairs, sl.cbase, sl.offset,
                                                             sl.n, p, ap, sc, turn);
          else if (quad) sv_spmv_it_quad<<<spmv_blocks, B, 0, s>>>(rp[0], ci[0], v[0], p, ap, na, sc, turn, v_bytes);
          else sv_spmv_it<<<spmv_blocks, B, 0, s>>>(rp[0], ci[0], v[0], p, ap, na, sc, turn);
          if (!fused) sv_dot_it<<<parts, B, 0, s>>>(p, ap, na, sc, turn, pc);
          if (precond == 0)
            sv_update_jacobi<<<parts, B, 0, s>>>(diag, p, ap, sc, turn, pc, na, x, r, z, pa, pb);
          else
            sv_update_block<<<parts, B, 0, s>>>(inv, starts, nblk, p, ap, sc, turn, pc, x, r, z, pa, pb);
          if (!fused || q + 1 == nq)
            sv_direction<<<parts, B, 0, s>>>(z, sc, turn, pa, pb, stop, double(max_iter), na, p);
        }
        HIP_TRY(hipGetLastError());
        const bool first = queued == 0;
        queued += nq;
        if (slice && first) {
          slice = slices_size(bufs, rp[0], ci[0], na, s, sl).empty();  // no memory: the solve goes on without
          if (slice) HIP_TRY(hipMemcpyAsync(host + S_COUNT, sl.offset + sl.n, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
          else (void)hipGetLastError();
        }
        HIP_TRY(hipMemcpyAsync(host, sc, sizeof(double) * S_COUNT, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        if (host[S_DONE] != 0.0 || host[S_DONE + 1] != 0.0 || queued >= max_iter) break;
        if (slice && first) {
          std::memcpy(&slice_total, host + S_COUNT, sizeof(uint32_t));
          slice = size_t(slice_total) * 256 <= SL_MAX_BYTES * size_t(d->sep_nnz[0]);
          if (slice && !slices_fill(bufs, rp[0], ci[0], v[0], v_bytes, slice_total, s, sl)) sl.data = nullptr;
        }
        batch = std::min(batch * 2, 64);
      }
      it = int(host[S_ITER]);
      conv = host[S_CONV] != 0.0;
    }
  }
  // r_r = (K_ba u_a + K_bb u_b) - r_b
  if (nb) {
    sv_gather<<<grid_for(nb, B), B, 0, s>>>(d->sep_force, bb_idx, nb, rb);
    sv_spmv<<<grid_for(nb * SPMV_LANES, B), B, 0, s>>>(rp[2], ci[2], v[2], x, nullptr, 1.0, nullptr, rr, nb);
    sv_spmv<<<grid_for(nb * SPMV_LANES, B), B, 0, s>>>(rp[3], ci[3], v[3], u_b, rr, 1.0, rb, rr, nb);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipEventRecord(d->ev5, s));
  HIP_TRY(hipStreamSynchronize(s));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, d->ev4, d->ev5));
  d->sol_ms = ms;
  res.iterations = it;
  res.converged = conv;
  res.residual = std::sqrt(host[S_RR]);
  res.stop = stop;
  return "";
}

// the model's own buffers, grown on demand
struct ModelBuffers : SolveBuffers {
  Device* d;
  explicit ModelBuffers(Device* dev) : d(dev) {}
  bool grows() const override { return true; }
  std::string get(int slot, size_t bytes, void** out) override {
    std::string e;
    const size_t n8 = (bytes + 7) / 8, n4 = (bytes + 3) / 4;
    if (slot < 6) { e = dgrow(d->sol_vec[slot], d->sol_cap[slot], n8); *out = d->sol_vec[slot]; }
    else if (slot == 6) { e = dgrow(d->sol_rr, d->sol_cap[6], n8); *out = d->sol_rr; }
    else if (slot == 7) { e = dgrow(d->sol_rb, d->sol_cap[7], n8); *out = d->sol_rb; }
    else if (slot == 8) { e = dgrow(d->sol_part, d->sol_cap[8], n8); *out = d->sol_part; }
    else if (slot == 9) { e = dgrow(d->sol_s, d->sol_cap[9], n8); *out = d->sol_s; }
    else if (slot == 10) { e = dgrow(d->sol_diag, d->sol_cap[10], n8); *out = d->sol_diag; }
    else if (slot == 11) { e = dgrow(d->sol_flag, d->sol_cap[11], n4); *out = d->sol_flag; }
    else if (slot == 12) { e = dgrow(d->sol_bid, d->sol_cap[12], n4); *out = d->sol_bid; }
    else if (slot == 13) { e = dgrow(d->sol_starts, d->sol_cap[13], n4); *out = d->sol_starts; }
    else if (slot == 14) { e = dgrow(d->sol_tmp, d->sol_cap[14], bytes); *out = d->sol_tmp; }
    else if (slot == 15) { e = dgrow(d->sol_inv, d->sol_cap[15], n8); *out = d->sol_inv; }
    else if (slot < 21) { e = dgrow(d->sol_slice[slot - 16], d->sol_cap[slot], n4); *out = d->sol_slice[slot - 16]; }
    else { e = dgrow(d->sol_slice_data, d->sol_cap[21], bytes); *out = d->sol_slice_data; }
    return e;
  }
};

}  // namespace

std::string solve_pcg(Device* d, int precond, int max_iter, double rel_tol, double abs_tol, void* stream,
                      SolveResult& res, bool wide, bool plain) {
  d->sol_done = false;
  if (!d->sep_done) return "no separation computed";
  if (!d->sol_host) HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&d->sol_host), 16 * sizeof(double)));
  ModelBuffers bufs(d);
  bufs.host = d->sol_host;
  auto e = solve_core(d, precond, max_iter, rel_tol, abs_tol, static_cast<hipStream_t>(stream), res, wide, plain, bufs);
  if (!e.empty()) return e;
  d->sol_na = d->sep_rows[0];
  d->sol_nb = d->sep_rows[2];
  d->sol_done = true;
  return "";
}

// ---- the solve without allocation: every work buffer in one static array per GPU

namespace {

static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

// device address of `scratch` on each GPU, looked up once per device (the
// array's name is only a host-side stand-in for it)
std::string scratch_address(void** out) {
  static std::mutex mu;
  static void* addr[64] = {};
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return "device index out of range for the static scratch table";
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return "hipGetSymbolAddress returned no address for the static scratch";
    addr[dev] = p;
  }
  *out = addr[dev];
  return "";
}

// slots 1 (u_a) and 6 (r_r) are the caller's outputs; the others are carved
// from the static array, each on a 256-byte boundary
struct StaticBuffers : SolveBuffers {
  unsigned char* base = nullptr;
  size_t used = 0;
  double *u_a = nullptr, *r_r = nullptr;
  size_t room() const override { return STATIC_SCRATCH_BYTES - std::min(STATIC_SCRATCH_BYTES, (used + 255) & ~size_t(255)); }
  std::string get(int slot, size_t bytes, void** out) override {
    if (slot == 1) { *out = u_a; return ""; }
    if (slot == 6) { *out = r_r; return ""; }
    const size_t off = (used + 255) & ~size_t(255);
    if (off + bytes > STATIC_SCRATCH_BYTES)
      return "the solve's work buffers exceed the static scratch of " + std::to_string(STATIC_SCRATCH_BYTES >> 20) +
             " MiB";
    *out = base + off;
    used = off + bytes;
    return "";
  }
};

}  // namespace

std::string solve_pcg_static(Device* d, int precond, int max_iter, double rel_tol, double abs_tol, void* stream,
                             double* u_a, double* r_r, SolveResult& res, bool wide, bool plain) {
  if (!d->sep_done) return "no separation computed";
  if ((!u_a && d->sep_rows[0]) || (!r_r && d->sep_rows[2])) return "u_a and r_r must be device buffers";
  void* base = nullptr;
  auto e = scratch_address(&base);
  if (!e.empty()) return e;
  StaticBuffers bufs;
  bufs.base = static_cast<unsigned char*>(base);
  bufs.u_a = u_a;
  bufs.r_r = r_r;
  double host[S_COUNT + 1];
  bufs.host = host;
  return solve_core(d, precond, max_iter, rel_tol, abs_tol, static_cast<hipStream_t>(stream), res, wide, plain, bufs);
}

std::string solution(Device* d, const double** u_a, const double** r_r, int64_t* n_aa, int64_t* n_bb) {
  if (!d->sol_done) return "no solution computed";
  if (u_a) *u_a = d->sol_vec[1];
  if (r_r) *r_r = d->sol_rr;
  if (n_aa) *n_aa = d->sol_na;
  if (n_bb) *n_bb = d->sol_nb;
  return "";
}

double last_solve_ms(Device* d) { return d->sol_ms; }

}  // namespace femdev
