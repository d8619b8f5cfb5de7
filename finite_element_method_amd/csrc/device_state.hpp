// device_state.hpp -- device-side state of one model, shared by the .hip files.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

namespace femdev {

struct UpdateReport;

// what the value path of the current pattern keeps of coordinates, frames and
// parameters in a form of its own: formed with its maps and by every update
enum class Kept { NONE, PLATE_SLOTS, FRAME_SLOTS, BAR_RECORDS };

// balanced-lane plate slots: their stride in doubles, and E, nu, k where every plate's are the same
struct PlateLaneHead {
  double mat[3];
  uint32_t stride;
};

struct Device {
  hipStream_t stream = nullptr;
  int dev = 0;
  double* xyz = nullptr;
  size_t n_nodes = 0;
  uint32_t* conn[3] = {nullptr, nullptr, nullptr};
  double* params[3] = {nullptr, nullptr, nullptr};
  double* R[3] = {nullptr, nullptr, nullptr};
  double* truss_dir = nullptr;  // trusses: R's first row, 3 doubles each (the only row the stiffness reads)
  double* derived = nullptr;  // beams: i11p, i22p
  uint16_t* rzero[3] = {nullptr, nullptr, nullptr};
  size_t n_elem[3] = {0, 0, 0};
  // CSR
  int64_t* row_ptr = nullptr;
  int32_t* col_idx = nullptr;
  double* val = nullptr;
  int64_t n_rows = 0, nnz = 0;
  Kept kept = Kept::NONE;
  // generic maps
  uint64_t* class_mask = nullptr;
  uint32_t* class_off = nullptr;
  uint16_t* eclass[3] = {nullptr, nullptr, nullptr};
  int64_t* ebase[3] = {nullptr, nullptr, nullptr};
  double* contrib = nullptr;
  int64_t n_contrib = 0;
  int64_t* slot_ptr = nullptr;
  uint32_t* slot_src = nullptr;
  // plate fused maps
  int n_patches = 0, pf_grid = 0, gen_block = 256;
  uint32_t *pf_hdr = nullptr, *pf_conn = nullptr, *pf_eid = nullptr, *pf_rows = nullptr, *pf_oinfo = nullptr,
           *pf_oboff = nullptr, *pf_oooff = nullptr, *pf_blk = nullptr;
  int64_t* pf_obase = nullptr;
  // plate block-lane maps
  int pb_patches = 0, pb_grid = 0;
  uint32_t *pb_hdr = nullptr, *pb_conn = nullptr, *pb_eid = nullptr, *pb_blk = nullptr;
  // plate balanced-lane maps (the element lists share pb_conn / pb_eid)
  int pl_waves = 0;
  uint32_t *pl_nodes = nullptr, *pl_lanes = nullptr, *pl_lane_set = nullptr;
  double* pl_geo = nullptr;   // per wave element slot: local coordinates and parameters
  // every plate has the same E, nu and k (bitwise): the slots hold t only and
  // the three values sit in the head
  bool pl_uniform = false;
  PlateLaneHead* pl_head = nullptr;
  // maps of plates in frames of their own (generic path of plate-only meshes);
  // pn_waves == 0: the generic path sums element contributions
  int pn_waves = 0;
  uint32_t *pn_eid = nullptr, *pn_nodes = nullptr, *pn_wave = nullptr, *pn_lanes = nullptr;
  double* pn_geo = nullptr;   // per wave element slot: local coordinates, parameters, frame
  // bar owner maps
  uint32_t* bo_bid[2] = {nullptr, nullptr};
  uint64_t* bo_bmask = nullptr;
  uint16_t* bo_boff = nullptr;
  uint32_t *bo_inc_ptr = nullptr, *bo_inc = nullptr, *bo_ranges = nullptr;
  size_t bo_n_ranges = 0, bo_n_truss_ranges = 0;  // bar-kernel ranges, then truss-kernel ranges
  int bo_truss_entries = 0;    // most entries of a truss-kernel range
  bool to_staged = false;      // truss ranges cut for the kernel that stages its rows
  uint32_t *bo_rec_elem = nullptr, *bo_entry_rec = nullptr, *bo_entry_ptr = nullptr;
  double* bo_rec = nullptr;    // element constants of the bar-kernel ranges
  uint4 *bo_entry = nullptr, *bo_self = nullptr;  // masks and row offsets: off-diagonal per entry, diagonal per node
  size_t bo_n_recs = 0;
  uint32_t *to_rec_elem = nullptr, *to_entry_rec = nullptr, *to_entry_ptr = nullptr;  // the truss kernel's
  double* to_rec = nullptr;
  uint4* to_entry = nullptr;
  size_t to_n_recs = 0;
  // adjoint maps
  uint32_t* adj_bid[3] = {nullptr, nullptr, nullptr};
  uint64_t* adj_bmask = nullptr;
  uint16_t* adj_boff = nullptr;
  uint32_t *adj_inc_ptr = nullptr, *adj_xpos = nullptr, *adj_kpack = nullptr;
  uint32_t* adj_eorder = nullptr;  // flat plates: elements in Morton order
  uint32_t* adj_beams = nullptr;   // beams likewise, four words each: the beam, its nodes, 0
  uint4* adj_rec[3] = {nullptr, nullptr, nullptr};  // per (element, node pair): its block's CSR positions and mask
  bool adj_rec_made = false;       // made (or left out for want of room) for these maps
  double* adj_xs = nullptr;
  int64_t adj_xoff[3] = {0, 0, 0};
  int64_t adj_nxs = 0;
  bool adj_flat = false;
  double rel_tol = 0.0, abs_tol = 0.0;
  // boundary conditions per global dof and the sparse separation; the four
  // matrices (K_aa, K_ab, K_ba, K_bb) share sep_rp / sep_ci / sep_v
  uint8_t *sep_cons = nullptr, *sep_cls = nullptr, *sep_tmp = nullptr;
  double *sep_disp = nullptr, *sep_force = nullptr, *sep_ra = nullptr, *sep_ub = nullptr, *sep_v = nullptr;
  uint64_t *sep_flag = nullptr, *sep_pos = nullptr;
  int64_t *sep_key = nullptr, *sep_cnt = nullptr, *sep_off = nullptr, *sep_aa = nullptr, *sep_bb = nullptr;
  int64_t *sep_rp = nullptr, *sep_sum = nullptr;
  int32_t* sep_ci = nullptr;
  int64_t* sep_dpos = nullptr;  // diagonal entry of each row (pattern-only)
  uint32_t* sep_pack = nullptr;  // per dof: class << 30 | its index among the a (or b) dofs
  uint8_t* sep_mark = nullptr;   // rows that hold a column that is not free
  uint8_t* sep_left = nullptr;   // groups of rows whose entries are not one run of K_aa
  uint64_t* sep_chunk = nullptr; // per chunk of dofs: a and b dofs (packed), then those before it
  uint32_t *sep_err = nullptr, *sep_rows2 = nullptr;  // per chunk its first error; per row its a and b entries
  int64_t* sep_host = nullptr;   // the summary, in pinned host memory
  bool sep_dpos_valid = false;
  size_t sep_cap[25] = {};
  int64_t sep_bc_rows = -1, sep_n_cons = 0;  // dofs of the uploaded boundary conditions, and restrained ones among them
  int64_t sep_rows[4] = {0, 0, 0, 0}, sep_nnz[4] = {0, 0, 0, 0}, sep_base[4] = {0, 0, 0, 0};
  bool sep_done = false;
  double sep_ms = 0.0;
  // sparse global analysis (solve.hip): b, x = u_a, r, z, p, Ap
  double* sol_vec[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  double *sol_rr = nullptr, *sol_rb = nullptr, *sol_part = nullptr, *sol_s = nullptr, *sol_host = nullptr;
  double *sol_diag = nullptr, *sol_inv = nullptr;
  uint32_t *sol_flag = nullptr, *sol_bid = nullptr;
  int32_t* sol_starts = nullptr;
  uint8_t* sol_tmp = nullptr;
  uint32_t* sol_slice[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};  // K_aa's slices: rows, pairs, lowest columns, sizes, offsets
  uint8_t* sol_slice_data = nullptr;                                       // and entries
  size_t sol_cap[22] = {};
  int64_t sol_na = 0, sol_nb = 0;
  bool sol_done = false;
  double sol_ms = 0.0;
  double* u_glob = nullptr;  // global displacements of the last solve (6 per node)
  size_t ucap = 0;
  // streams that were given work since the last update that reads what an update
  // rewrites (note_use; of more than two, two say enough); captured: such work is
  // in a graph, whose replays may run on any stream
  hipStream_t used[2] = {nullptr, nullptr};
  int n_used = 0;
  bool captured = false;
  // updates in place (fem_device.hip): report words, their copy in pinned host
  // memory, and the number of the last update
  uint32_t* upd_words = nullptr;
  UpdateReport* upd_report = nullptr;
  uint32_t upd_number = 0;
  // timing
  hipEvent_t ev0 = nullptr, ev1 = nullptr, ev2 = nullptr, ev3 = nullptr, ev4 = nullptr, ev5 = nullptr;
  bool timed = false, timed_bwd = false;
};

#define HIP_TRY(expr)                                                                 \
  do {                                                                                \
    hipError_t _e = (expr);                                                           \
    if (_e != hipSuccess) return std::string(#expr) + ": " + hipGetErrorString(_e);  \
  } while (0)

// form what the path keeps (Kept) from the current coordinates, frames and parameters
std::string plate_lanes_gather(Device* d, hipStream_t s);   // plate_lanes.hip
std::string plate_frames_gather(Device* d, hipStream_t s);  // plate_frames.hip
std::string fill_bar_records(Device* d, hipStream_t s);     // bar_owner.hip

template <class T>
inline std::string dalloc(T*& p, size_t n) {
  if (p) { (void)hipFree(p); p = nullptr; }
  if (n == 0) return "";
  HIP_TRY(hipMalloc(&p, n * sizeof(T)));
  return "";
}
template <class T>
inline std::string dupload(T*& p, const T* src, size_t n) {
  auto e = dalloc(p, n);
  if (!e.empty()) return e;
  if (n) HIP_TRY(hipMemcpy(p, src, n * sizeof(T), hipMemcpyHostToDevice));
  return "";
}

}  // namespace femdev
