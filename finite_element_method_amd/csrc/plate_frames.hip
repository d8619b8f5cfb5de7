// plate_frames.hip -- assembly of plate meshes whose elements have frames of
// their own (shells, tilted plates): one wave per patch of owned nodes, one lane
// per owned node-pair block, values staged in LDS and written out as
// consecutive 16-byte chunks.
//
// The value path of such meshes that needs no buffer of element contributions:
// every owned block is summed in registers, in element-insertion order
// (methods_for_plate_data_handle.rs:134-212), from records that the wave forms
// for the elements touching its nodes, and each CSR value is written once.
//
// Steps of a wave:
//   1. element records: four lanes per element, one integration point each, form
//      the point's share of the 42 integrals of every node-pair bilinear form
//      and add the four shares by two DPP exchanges, after which each lane holds
//      and writes its own quarter; the frame R and the constants go along;
//   2. blocks: each lane sums its block over the elements that hold both nodes:
//      13 local entries from the record (record_block), turned to the global
//      axes by their structure (R^T k R of methods_for_plate_data_handle.rs:104-112
//      without the products of k's zeros);
//   3. staging: the block's structural entries go to their places in the node's
//      CSR rows in LDS, which reuses the records' space;
//   4. copy-out by runs of nodes whose rows follow each other, non-temporal
//      16-byte stores of whole aligned groups, as plate_lanes.hip.
//
// Bound: the value stores.  A node of a regular shell has 9 blocks of 36 values
// (2592 bytes) against 54 bytes of coordinates, connectivity and parameters per
// element; the arithmetic (about 8 kFLOP per element) overlaps them.
// 64 lanes hold the blocks of seven such nodes, whose strip of the mesh touches
// 16 elements: 16 x 4 record lanes and 63 block lanes, 18.6 KB of LDS.
// Measured on a shell of 301 x 217 elements (174 MB of compulsory traffic, 35 us
// at the rate of a large copy): 51 us, 3.4 TB/s; through the buffer of element
// contributions (generic_items_kernel, slot_gather_kernel) 418 us.
#include <hip/hip_runtime.h>

#include "device_state.hpp"
#include "element_math.hpp"
#include "fem_device.hpp"
#include "plate_record.hpp"

namespace femdev {

namespace {

typedef unsigned int pn_u32x4 __attribute__((ext_vector_type(4)));

constexpr int R_ROT = R_MAT + 6;     // the frame follows the plate record's constants
constexpr int PN_REC = R_ROT + 10;   // doubles; 16-byte records, 4 banks apart
constexpr int PN_GEO = 20;           // element slot: x1, y1, x2, y2, x4, y4 in the frame; E, nu, t, k; R; pad
constexpr int PN_STORE_NT = 2;       // buffer-store cache policy: non-temporal
constexpr int PN_LDS = PN_ELEMS * PN_REC > PN_STAGE_VALUES ? PN_ELEMS * PN_REC : PN_STAGE_VALUES;
static_assert(PN_REC % 2 == 0 && PN_LDS % 2 == 0, "16-byte records");
static_assert(4 * PN_ELEMS == 64, "four lanes per element");

struct FrameArgs {
  const double* __restrict__ geo;     // per wave PN_ELEMS slots of PN_GEO doubles
  const uint2* __restrict__ nodes;    // per wave PN_NODES: CSR position of row 6a, staging position | values << 12
  const uint2* __restrict__ waves;    // per wave: descriptor set, elements | nodes << 8 | trips << 16
  const uint4* __restrict__ lanes;    // per set 64 x 2: see PlateFrameMaps
  double* __restrict__ val;
  uint32_t val_bytes;
};

// Element slots: local coordinates of nodes 1, 2, 4 about node 3 in the
// element's frame (quad:340-378), the parameters and the frame.
__global__ __launch_bounds__(256) void plate_frames_gather_kernel(const double* __restrict__ xyz,
                                                                  const uint32_t* __restrict__ conn,
                                                                  const double* __restrict__ params,
                                                                  const double* __restrict__ Rall,
                                                                  const uint32_t* __restrict__ seid, size_t n_slots,
                                                                  double* __restrict__ geo) {
  const size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (i >= n_slots) return;
  const uint32_t e = seid[i];
  double2* g = reinterpret_cast<double2*>(geo + i * PN_GEO);
  if (e == 0xFFFFFFFFu) {  // unused slot: never read as an element
    for (int k = 0; k < PN_GEO / 2; ++k) g[k] = make_double2(0.0, 0.0);
    return;
  }
  const uint4 c = *reinterpret_cast<const uint4*>(conn + 4 * size_t(e));
  const uint32_t n[4] = {c.x, c.y, c.z, c.w};
  double R[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) R[k] = Rall[9 * size_t(e) + k];
  double X[4][3];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int k = 0; k < 3; ++k) X[a][k] = xyz[3 * size_t(n[a]) + k];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int a = m < 2 ? m : 3;
    const double d[3] = {X[a][0] - X[2][0], X[a][1] - X[2][1], X[a][2] - X[2][2]};
    g[m] = make_double2((R[0] * d[0] + R[1] * d[1]) + R[2] * d[2], (R[3] * d[0] + R[4] * d[1]) + R[5] * d[2]);
  }
  const double* p = params + 4 * size_t(e);
  g[3] = make_double2(p[0], p[1]);
  g[4] = make_double2(p[2], p[3]);
#pragma unroll
  for (int k = 0; k < 4; ++k) g[5 + k] = make_double2(R[2 * k], R[2 * k + 1]);
  g[9] = make_double2(R[8], 0.0);
}

// both 32-bit halves of a double from lane ^ 2, by DPP
__device__ inline double swap_pairs(double v) {
  const pl_u32x2 x = __builtin_bit_cast(pl_u32x2, v);
  pl_u32x2 r;
  r.x = uint32_t(__builtin_amdgcn_mov_dpp(int(x.x), 0x4E, 0xF, 0xF, false));
  r.y = uint32_t(__builtin_amdgcn_mov_dpp(int(x.y), 0x4E, 0xF, 0xF, false));
  return __builtin_bit_cast(double, r);
}

// acc += R6^T k R6 of the local block k given by its 13 entries o and, on
// diagonal blocks, the drilling stiffness kd: with r0, r1 the in-plane rows of R
// and n its normal row,
//   translations:        membrane 2x2 in (r0, r1), (w, w) on n n^T
//   translation-rotation: n (x) ((w,tx) r0 + (w,ty) r1), and its mirror
//   rotations:           bending + shear 2x2 in (r0, r1), kd on n n^T
__device__ inline void add_rotated(const double o[13], double kd, const double* R, double acc[36]) {
  const double2 q0 = *reinterpret_cast<const double2*>(R), q1 = *reinterpret_cast<const double2*>(R + 2),
                q2 = *reinterpret_cast<const double2*>(R + 4), q3 = *reinterpret_cast<const double2*>(R + 6);
  const double r0[3] = {q0.x, q0.y, q1.x}, r1[3] = {q1.y, q2.x, q2.y}, n[3] = {q3.x, q3.y, R[8]};
  double m0[3], m1[3], b0[3], b1[3], s[3], z[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    m0[j] = o[0] * r0[j] + o[1] * r1[j];    // membrane rows u, v
    m1[j] = o[2] * r0[j] + o[3] * r1[j];
    s[j] = o[5] * r0[j] + o[6] * r1[j];     // row w against the rotations
    z[j] = o[7] * r0[j] + o[10] * r1[j];    // column w against the rotations
    b0[j] = o[8] * r0[j] + o[9] * r1[j];    // rows tx, ty
    b1[j] = o[11] * r0[j] + o[12] * r1[j];
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const double wn = o[4] * n[i], kn = kd * n[i];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      acc[6 * i + j] += (r0[i] * m0[j] + r1[i] * m1[j]) + wn * n[j];
      acc[6 * i + 3 + j] += n[i] * s[j];
      acc[6 * (3 + i) + j] += z[i] * n[j];
      acc[6 * (3 + i) + 3 + j] += (r0[i] * b0[j] + r1[i] * b1[j]) + kn * n[j];
    }
  }
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void plate_frames_kernel(FrameArgs A) {
  // element records during steps 1-2, the owned nodes' staged values after
  __shared__ double2 lds2[PN_LDS / 2];
  double* rec = reinterpret_cast<double*>(lds2);
  double* stage = rec;
  const int l = threadIdx.x;
  const int le = l >> 2, ip = l & 3;
  const uint32_t w = blockIdx.x;
  const uint2 wave = A.waves[w];
  const int nel = int(wave.y & 255u), nnod = int((wave.y >> 8) & 255u), trips = int(wave.y >> 16);
  const double2* gs = reinterpret_cast<const double2*>(A.geo + (size_t(w) * PN_ELEMS + le) * PN_GEO);
  const double2 g0 = gs[0], g1 = gs[1], g2 = gs[2], g3 = gs[3 + 2 * ip], g4 = gs[ip == 3 ? 9 : 4 + 2 * ip];
  const uint4* ds = A.lanes + (size_t(wave.x) * 64 + l) * 2;
  const uint4 d0 = ds[0], d1 = ds[1];
  const uint2 nd = A.nodes[size_t(w) * PN_NODES + (l & (PN_NODES - 1))];

  // ---- step 1: element records, one integration point per lane
  {
    const bool live = le < nel;
    double I[PL_NINT];
#pragma unroll
    for (int k = 0; k < PL_NINT; ++k) I[k] = 0.0;
    const double xl[6] = {g0.x, g0.y, g1.x, g1.y, g2.x, g2.y};
    if (live) {
      fem::PlatePoint g;
      fem::plate_point(xl, ip, g);
      double wdx[4], wdy[4];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        wdx[a] = g.w * g.dx[a];
        wdy[a] = g.w * g.dy[a];
      }
      int s = 0;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = a; b < 4; ++b, ++s) {
          I[s] = wdx[a] * g.dx[b];
          I[R_MYY + s] = wdy[a] * g.dy[b];
        }
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) I[R_MXY + 4 * a + b] = wdx[a] * g.dy[b];
      const double al0 = g.al[0], al1 = g.al[2], be0 = g.be[0], be1 = g.be[1];
      const double wal0 = g.w * al0, wal1 = g.w * al1, wbe0 = g.w * be0, wbe1 = g.w * be1;
      I[R_A + 0] = wal0 * al0;
      I[R_A + 1] = wal0 * al1;
      I[R_A + 2] = wal1 * al1;
      // beta classes {0, 3} | {1, 2}
      I[R_B + 0] = wbe0 * be0;
      I[R_B + 1] = wbe0 * be1;
      I[R_B + 2] = wbe1 * be1;
    }
    // (point 0 + point 1) + (point 2 + point 3): lane bit 0 keeps integrals
    // 21 h .., lane bit 1 then 11 (of its 21) or the other 10
    const bool h = ip & 1, b = ip & 2;
    double S[PL_NINT / 2], T[11];
#pragma unroll
    for (int k = 0; k < PL_NINT / 2; ++k) {
      const double mine = h ? I[k + PL_NINT / 2] : I[k];
      S[k] = mine + swap_pair(h ? I[k] : I[k + PL_NINT / 2]);
    }
#pragma unroll
    for (int k = 0; k < 11; ++k) {
      const double up = k < 10 ? S[k + 11] : 0.0;
      T[k] = (b ? up : S[k]) + swap_pairs(b ? S[k] : up);
    }
    if (live) {
      double* r = rec + le * PN_REC;
      double* t = r + (h ? 21 : 0) + (b ? 11 : 0);
#pragma unroll
      for (int k = 0; k < 10; ++k) t[k] = T[k];
      if (!b) t[10] = T[10];
      // shear edge vectors (plate.rs:452-508): e12, e43, e14, e23, one per lane
      const double ex = ip == 0 ? xl[0] - xl[2] : ip == 1 ? xl[4] : ip == 2 ? xl[0] - xl[4] : xl[2];
      const double ey = ip == 0 ? xl[1] - xl[3] : ip == 1 ? xl[5] : ip == 2 ? xl[1] - xl[5] : xl[3];
      *reinterpret_cast<double2*>(r + R_SH + 2 * ip) = make_double2(-ey * 0.25, ex * 0.25);
      if (ip == 0) {
        const fem::PlateMat mt = fem::plate_material(g3.x, g3.y, g4.x, g4.y);
        // bending constants are the membrane ones times t^2 / 12 (plate.rs:532-636)
        const double tb = (g4.x * g4.x) / 12.0;
        *reinterpret_cast<double2*>(r + R_MAT) = make_double2(mt.cm00, mt.cm01);
        *reinterpret_cast<double2*>(r + R_MAT + 2) = make_double2(mt.cm22, tb);
        *reinterpret_cast<double2*>(r + R_MAT + 4) = make_double2(mt.cs, 0.0);
      } else {  // R: lane 1 elements 0..3, lane 2 4..7, lane 3 the last (g3 == g4)
        double2* rr = reinterpret_cast<double2*>(r + R_ROT + 4 * (ip - 1));
        rr[0] = g3;
        if (ip < 3) rr[1] = g4;
      }
    }
  }
  wave_lds_sync();

  // ---- step 2: blocks in element-insertion order.  Items of 8 bits: wave
  // element | p << 4 | q << 6
  const uint64_t items = uint64_t(d0.x) | uint64_t(d0.y) << 32;
  const uint64_t mask = uint64_t(d0.z) | uint64_t(d0.w & 15u) << 32;
  const int cnt = int((d0.w >> 4) & 15u);
  double acc[36];
#pragma unroll
  for (int k = 0; k < 36; ++k) acc[k] = 0.0;
  for (int t = 0; t < trips; ++t) {
    if (t < cnt) {
      const uint32_t it = uint32_t(items >> (8 * t)) & 255u;
      const int p = int((it >> 4) & 3u), q = int(it >> 6);
      const double* r = rec + int(it & 15u) * PN_REC;
      double o[13];
      record_block(r, p, q, o);
      add_rotated(o, p == q ? fem::KROT6 : 0.0, r + R_ROT, acc);
    }
  }
  wave_lds_sync();  // every record read is done: the staging reuses the records' LDS

  // ---- step 3: structural entries to their places in the node's rows
  if (cnt) {
    const uint32_t off[6] = {d1.x & 0xFFFFu, d1.x >> 16, d1.y & 0xFFFFu, d1.y >> 16, d1.z & 0xFFFFu, d1.z >> 16};
    const uint32_t odd = (off[0] | off[1] | off[2] | off[3] | off[4] | off[5]) & 1u;
    if (mask == 0xFFFFFFFFFull && !odd) {  // a full block at even positions: 16-byte stores
#pragma unroll
      for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; j += 2)
          *reinterpret_cast<double2*>(stage + off[i] + j) = make_double2(acc[6 * i + j], acc[6 * i + j + 1]);
    } else {
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        uint32_t o = off[i];
#pragma unroll
        for (int j = 0; j < 6; ++j)
          if ((mask >> (6 * i + j)) & 1ull) stage[o++] = acc[6 * i + j];
      }
    }
  }
  wave_lds_sync();

  // ---- step 4: copy-out by runs of owned nodes whose CSR ranges follow each
  // other (staged contiguously, at the CSR parity); non-temporal
  const double2* stage2 = lds2;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(A.val, 0, int(A.val_bytes), 0x00020000);
  int s0 = 0;
  while (s0 < nnod) {
    const uint32_t base = uint32_t(__builtin_amdgcn_readlane(int(nd.x), s0));
    const uint32_t w0 = uint32_t(__builtin_amdgcn_readlane(int(nd.y), s0));
    uint32_t end = base + (w0 >> 12);
    int s1 = s0 + 1;
    while (s1 < nnod && uint32_t(__builtin_amdgcn_readlane(int(nd.x), s1)) == end) {
      end += uint32_t(__builtin_amdgcn_readlane(int(nd.y), s1)) >> 12;
      ++s1;
    }
    const int shift = int((w0 & 0xFFFu) >> 1) - int(base >> 1);  // staging chunk - CSR chunk (same parity)
    for (uint32_t c = ((base >> 1) & ~7u) + uint32_t(l); c < (end + 1u) >> 1; c += 64u) {
      if (c < (base >> 1)) continue;
      const double2 v = stage2[int(c) + shift];
      const uint32_t g = 2u * c;  // first value of the chunk
      if (g >= base && g + 1u < end) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(pn_u32x4, v), rsrc, 8u * g, 0, PN_STORE_NT);
      } else if (g < base) {  // the run starts at an odd position: the chunk's upper half
        if (g + 1u < end)
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(pl_u32x2, v.y), rsrc, 8u * g + 8u, 0, PN_STORE_NT);
      } else {  // the run ends at an odd position: the chunk's lower half
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(pl_u32x2, v.x), rsrc, 8u * g, 0, PN_STORE_NT);
      }
    }
    s0 = s1;
  }
}

}  // namespace

std::string plate_frames_gather(Device* d, hipStream_t s) {
  const size_t n_slots = size_t(d->pn_waves) * PN_ELEMS;
  if (n_slots) {
    plate_frames_gather_kernel<<<unsigned((n_slots + 255) / 256), 256, 0, s>>>(d->xyz, d->conn[PLATE], d->params[PLATE],
                                                                             d->R[PLATE], d->pn_eid, n_slots, d->pn_geo);
    HIP_TRY(hipGetLastError());
  }
  return "";
}

std::string upload_plate_frame_maps(Device* d, const PlateFrameMaps& pm) {
  d->pn_waves = 0;
  std::string e;
  if (!(e = dupload(d->pn_eid, pm.seid.data(), pm.seid.size())).empty()) return e;
  if (!(e = dupload(d->pn_nodes, pm.nodes.data(), pm.nodes.size())).empty()) return e;
  if (!(e = dupload(d->pn_lanes, pm.lanes.data(), pm.lanes.size())).empty()) return e;
  if (!(e = dupload(d->pn_wave, pm.waves.data(), pm.waves.size())).empty()) return e;
  if (!(e = dalloc(d->pn_geo, size_t(pm.n_waves) * PN_ELEMS * PN_GEO)).empty()) return e;
  d->pn_waves = pm.n_waves;
  if (!(e = plate_frames_gather(d, nullptr)).empty()) return e;
  d->kept = Kept::FRAME_SLOTS;
  HIP_TRY(hipDeviceSynchronize());
  return "";
}

std::string assemble_plate_frames(Device* d, double* val, void* stream, bool timed) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (timed) HIP_TRY(hipEventRecord(d->ev0, s));
  FrameArgs a;
  a.geo = d->pn_geo;
  a.nodes = reinterpret_cast<const uint2*>(d->pn_nodes);
  a.waves = reinterpret_cast<const uint2*>(d->pn_wave);
  a.lanes = reinterpret_cast<const uint4*>(d->pn_lanes);
  a.val = val;
  a.val_bytes = uint32_t(d->nnz * 8);
  plate_frames_kernel<<<unsigned(d->pn_waves), 64, 0, s>>>(a);
  HIP_TRY(hipGetLastError());
  if (timed) {
    HIP_TRY(hipEventRecord(d->ev1, s));
    d->timed = true;
  }
  return "";
}

}  // namespace femdev
