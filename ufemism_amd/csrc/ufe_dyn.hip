// ufe_dyn.hip -- context, device layouts, drivers and the C-ABI of libufe_dyn.
//
// The reference runs its ice-dynamics loops on MPI ranks sharing memory
// windows (src/parallel_module.f90).  Here one context owns device-resident
// copies of the mesh and of every ice-model field, and each reference routine
// becomes a short sequence of kernels on the context's stream.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "ufe_internal.h"
#include <hip/hip_ext.h>
#include <type_traits>

#include "amg_host.h"
#include "patch_host.h"
#include "ufe_kernels.inc"
#include "patch_kernels.inc"

namespace ufe {

// ---------------------------------------------------------------------------
// Field table (type_ice_model subset, src/data_types_module.f90:15-214)
// ---------------------------------------------------------------------------
enum Grid { G_AA = 0, G_AAZ = 1, G_AAC = 2, G_AC = 3, G_ACZ = 4, G_AAAC = 5 };
enum DType { D_F64 = 0, D_I32 = 1 };
struct FieldDef {
  const char *name;
  int grid, dtype;
  int pair;    // -1, or index of an interleaved double2 store (0 W, 1 EV, 2 RHS)
  int comp;
};

static const FieldDef FIELDS[] = {
    // Aa
    {"Hi", G_AA, D_F64, -1, 0}, {"Hb", G_AA, D_F64, -1, 0}, {"SL", G_AA, D_F64, -1, 0},
    {"Hs", G_AA, D_F64, -1, 0}, {"dHb_dt", G_AA, D_F64, -1, 0}, {"dHi_dt", G_AA, D_F64, -1, 0},
    {"dHs_dt", G_AA, D_F64, -1, 0}, {"Hi_prev", G_AA, D_F64, -1, 0},
    {"A_flow_mean", G_AA, D_F64, -1, 0}, {"dHi_dx", G_AA, D_F64, -1, 0},
    {"dHi_dy", G_AA, D_F64, -1, 0}, {"dHs_dx", G_AA, D_F64, -1, 0}, {"dHs_dy", G_AA, D_F64, -1, 0},
    {"dHs_dx_shelf", G_AA, D_F64, -1, 0}, {"dHs_dy_shelf", G_AA, D_F64, -1, 0},
    {"U_SIA", G_AA, D_F64, -1, 0}, {"V_SIA", G_AA, D_F64, -1, 0}, {"D_SIA", G_AA, D_F64, -1, 0},
    {"U_SSA", G_AA, D_F64, -1, 0}, {"V_SSA", G_AA, D_F64, -1, 0},
    {"SMB_year", G_AA, D_F64, -1, 0}, {"BMB", G_AA, D_F64, -1, 0},
    {"A_flow", G_AAZ, D_F64, -1, 0}, {"Ti", G_AAZ, D_F64, -1, 0}, {"Ti_pmp", G_AAZ, D_F64, -1, 0},
    {"Cpi", G_AAZ, D_F64, -1, 0}, {"Ki", G_AAZ, D_F64, -1, 0}, {"U_3D", G_AAZ, D_F64, -1, 0},
    {"V_3D", G_AAZ, D_F64, -1, 0}, {"W_3D", G_AAZ, D_F64, -1, 0}, {"dVi_in", G_AAC, D_F64, -1, 0},
    // Ac
    {"Hi_Ac", G_AC, D_F64, -1, 0}, {"Hb_Ac", G_AC, D_F64, -1, 0}, {"SL_Ac", G_AC, D_F64, -1, 0},
    {"Hs_Ac", G_AC, D_F64, -1, 0},
    {"dHi_dx_Ac", G_AC, D_F64, -1, 0}, {"dHi_dy_Ac", G_AC, D_F64, -1, 0},
    {"dHi_dp_Ac", G_AC, D_F64, -1, 0}, {"dHi_do_Ac", G_AC, D_F64, -1, 0},
    {"dHb_dx_Ac", G_AC, D_F64, -1, 0}, {"dHb_dy_Ac", G_AC, D_F64, -1, 0},
    {"dHb_dp_Ac", G_AC, D_F64, -1, 0}, {"dHb_do_Ac", G_AC, D_F64, -1, 0},
    {"dHs_dx_Ac", G_AC, D_F64, -1, 0}, {"dHs_dy_Ac", G_AC, D_F64, -1, 0},
    {"dHs_dp_Ac", G_AC, D_F64, -1, 0}, {"dHs_do_Ac", G_AC, D_F64, -1, 0},
    {"dSL_dx_Ac", G_AC, D_F64, -1, 0}, {"dSL_dy_Ac", G_AC, D_F64, -1, 0},
    {"dSL_dp_Ac", G_AC, D_F64, -1, 0}, {"dSL_do_Ac", G_AC, D_F64, -1, 0},
    {"dHs_dx_shelf_Ac", G_AC, D_F64, -1, 0}, {"dHs_dy_shelf_Ac", G_AC, D_F64, -1, 0},
    {"A_flow_mean_Ac", G_AC, D_F64, -1, 0},
    {"D_SIA_Ac", G_AC, D_F64, -1, 0}, {"Ux_SIA_Ac", G_AC, D_F64, -1, 0},
    {"Uy_SIA_Ac", G_AC, D_F64, -1, 0}, {"Up_SIA_Ac", G_AC, D_F64, -1, 0},
    {"Uo_SIA_Ac", G_AC, D_F64, -1, 0}, {"Ux_SSA_Ac", G_AC, D_F64, -1, 0},
    {"Uy_SSA_Ac", G_AC, D_F64, -1, 0}, {"Up_SSA_Ac", G_AC, D_F64, -1, 0},
    {"Uo_SSA_Ac", G_AC, D_F64, -1, 0},
    {"Qabs_GL_Ac", G_AC, D_F64, -1, 0}, {"Qp_GL_Ac", G_AC, D_F64, -1, 0},
    {"A_flow_Ac", G_ACZ, D_F64, -1, 0}, {"D_SIA_3D_Ac", G_ACZ, D_F64, -1, 0},
    {"Ti_Ac", G_ACZ, D_F64, -1, 0},
    // AaAc (stored in colour order)
    {"Hi_AaAc", G_AAAC, D_F64, -1, 0}, {"Hb_AaAc", G_AAAC, D_F64, -1, 0},
    {"SL_AaAc", G_AAAC, D_F64, -1, 0}, {"dHs_dx_shelf_AaAc", G_AAAC, D_F64, -1, 0},
    {"dHs_dy_shelf_AaAc", G_AAAC, D_F64, -1, 0}, {"A_flow_mean_AaAc", G_AAAC, D_F64, -1, 0},
    {"U_SSA_AaAc", G_AAAC, D_F64, 0, 0}, {"V_SSA_AaAc", G_AAAC, D_F64, 0, 1},
    {"dU_SSA_dx_AaAc", G_AAAC, D_F64, -1, 0}, {"dU_SSA_dy_AaAc", G_AAAC, D_F64, -1, 0},
    {"dV_SSA_dx_AaAc", G_AAAC, D_F64, -1, 0}, {"dV_SSA_dy_AaAc", G_AAAC, D_F64, -1, 0},
    {"eta_AaAc", G_AAAC, D_F64, -1, 0}, {"N_AaAc", G_AAAC, D_F64, -1, 0},
    {"N_AaAc_prev", G_AAAC, D_F64, -1, 0}, {"S_AaAc", G_AAAC, D_F64, -1, 0},
    {"phi_fric_AaAc", G_AAAC, D_F64, -1, 0}, {"tau_c_AaAc", G_AAAC, D_F64, -1, 0},
    {"RHSx_AaAc", G_AAAC, D_F64, 2, 0}, {"RHSy_AaAc", G_AAAC, D_F64, 2, 1},
    {"eu_i_AaAc", G_AAAC, D_F64, 1, 0}, {"ev_i_AaAc", G_AAAC, D_F64, 1, 1},
    {"tau_c_override_AaAc", G_AAAC, D_F64, -1, 0},
    // masks
    {"mask_land", G_AA, D_I32, -1, 0}, {"mask_ocean", G_AA, D_I32, -1, 0},
    {"mask_lake", G_AA, D_I32, -1, 0}, {"mask_ice", G_AA, D_I32, -1, 0},
    {"mask_sheet", G_AA, D_I32, -1, 0}, {"mask_shelf", G_AA, D_I32, -1, 0},
    {"mask_coast", G_AA, D_I32, -1, 0}, {"mask_margin", G_AA, D_I32, -1, 0},
    {"mask_gl", G_AA, D_I32, -1, 0}, {"mask_cf", G_AA, D_I32, -1, 0}, {"mask", G_AA, D_I32, -1, 0},
    {"mask_land_Ac", G_AC, D_I32, -1, 0}, {"mask_ocean_Ac", G_AC, D_I32, -1, 0},
    {"mask_lake_Ac", G_AC, D_I32, -1, 0}, {"mask_ice_Ac", G_AC, D_I32, -1, 0},
    {"mask_sheet_Ac", G_AC, D_I32, -1, 0}, {"mask_shelf_Ac", G_AC, D_I32, -1, 0},
    {"mask_coast_Ac", G_AC, D_I32, -1, 0}, {"mask_margin_Ac", G_AC, D_I32, -1, 0},
    {"mask_gl_Ac", G_AC, D_I32, -1, 0}, {"mask_cf_Ac", G_AC, D_I32, -1, 0},
    {"mask_Ac", G_AC, D_I32, -1, 0}, {"mask_noice", G_AA, D_I32, -1, 0},
};
static const int NFIELDS = (int)(sizeof(FIELDS) / sizeof(FIELDS[0]));

static int field_id(const char *name) {
  for (int i = 0; i < NFIELDS; i++)
    if (std::strcmp(FIELDS[i].name, name) == 0) return i;
  return -1;
}

template <typename T>
struct DevBuf {
  T *p = nullptr;
  size_t n = 0;
};

}  // namespace ufe

using namespace ufe;

// One coarse level of the aggregation multigrid preconditioner (device arrays;
// allocated with the mesh).  Level 1 aggregates the SOR rows of the fine
// operator, level l + 1 the points of level l.
struct AmgLevel {
  int n = 0;                        // points
  int64_t nnz = 0;
  int32_t *ptr = nullptr, *col = nullptr;   // off-diagonal couplings, CSR over points
  float2 *cf = nullptr;
  int32_t *ptrT = nullptr, *colT = nullptr; // the transposed couplings (adjoint solves)
  float2 *cfT = nullptr;
  float *S = nullptr;               // u-v coupling of each point with itself
  double2 *fd = nullptr;            // diagonal pair added to the members' diagonals (fixed per mesh)
  double2 *ev64 = nullptr;          // diagonal pair of the current system
  float2 *ev32 = nullptr;
  int32_t *mptr = nullptr, *mem = nullptr;  // members: rows of the fine level (level 1) or points above
  int32_t *agg = nullptr;           // row / point above -> this level's point (-1: not aggregated)
  int nmem = 0, nagg = 0;           // lengths of mem and agg
  float2 *ev32_img = nullptr;       // ev32's place in the small-level kernel's image, or null
  bool blocks = false;              // F holds the fused kernels' blocks and halos (K-step dots by block)
  bool fuse = false;                // cycle steps by k_amg_fuse_pre / k_amg_fuse_post
  AmgFuse F{};
  int fuse_blocks = 0;
  bool fuseT = false;               // and for the transposed operator: its local rows
  int32_t *fuse_rptrT = nullptr;
  uint16_t *fuse_lcolT = nullptr;
  float2 *fuse_lcfT = nullptr;
  float2 *b = nullptr, *t = nullptr, *e1 = nullptr, *e2 = nullptr, *w1 = nullptr, *w2 = nullptr,
         *rc2 = nullptr, *r = nullptr;
  double *part = nullptr, *sc = nullptr;
  double2 *cf64 = nullptr;          // coarsest level: FP64 couplings for the dense inverse
  double *S64 = nullptr;
  bool kstep = false;               // solved by two cycles with a GCR(2) combination
};

// A set of patches on the device (patch_host.h), built on first use per mesh.
enum PatchKind { PATCH_PRE32 = 0, PATCH_POST32, PATCH_SOR64, PATCH_KINDS };
struct PatchSet {
  bool built = false, ok = false;   // ok: the mesh fits (otherwise the per-colour kernels run)
  int bs = 0;                       // threads per workgroup
  size_t lds = 0;
  PatchDev P{};
};

struct ufe_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  ufe_params params{};
  bool have_mesh = false;
  // sizes
  int nV = 0, nTri = 0, nCm = 0, nAc = 0, nA = 0, nZ = 15;
  // Aa / Ac mesh (reference layout on the device)
  int32_t *d_nC = nullptr, *d_C = nullptr, *d_edge = nullptr, *d_iAci = nullptr, *d_Crev = nullptr;
  double *d_Nx = nullptr, *d_Ny = nullptr, *d_Nxx = nullptr, *d_Nxy = nullptr, *d_Nyy = nullptr;
  double *d_A = nullptr, *d_Cw = nullptr, *d_V = nullptr;
  // triangles: upwind derivatives (Tri, iTri, triangle neighbour functions, resolution)
  int32_t *d_Tri = nullptr, *d_niTri = nullptr, *d_iTri = nullptr;
  double *d_NxTri = nullptr, *d_NyTri = nullptr, *d_R = nullptr;
  double *d_crit = nullptr;          // critical time step partial minima
  // remapping arrays from another context's mesh onto this one (ufe_remap_build)
  bool rm_ready = false;
  int rm_nVs = 0, rm_nVd = 0, rm_n = 0;
  int32_t *d_rm_nn = nullptr, *d_rm_tvi = nullptr, *d_rm_st = nullptr, *d_rm_en = nullptr, *d_rm_vi = nullptr;
  double *rm_work = nullptr;         // source derivatives of a second-order remapping (not in allocs: it grows)
  size_t rm_work_len = 0;
  double *d_rm_tw = nullptr, *d_rm_w0 = nullptr, *d_rm_w1x = nullptr, *d_rm_w1y = nullptr;
  int32_t *d_icount = nullptr;       // small device counters (upwind misses)
  int32_t *d_Aci = nullptr, *d_edgeAc = nullptr, *d_slot_i = nullptr, *d_slot_j = nullptr;
  double *d_NxAc = nullptr, *d_NyAc = nullptr, *d_NoAc = nullptr, *d_NpAc = nullptr;
  // AaAc colour order
  int32_t *d_perm = nullptr, *d_iperm = nullptr;
  std::vector<int32_t> h_perm;
  std::vector<uint32_t> h_key;      // Hilbert key of each row
  std::vector<uint16_t> h_mid;      // batch member of each row (empty: single mesh)
  PatchSet patch[PATCH_KINDS][2];   // by kind and sweeps - 1
  double2 *sor_w1 = nullptr;        // second buffer of the SOR loop on patches
  double2 *sor_start = nullptr;     // and the velocities that its launch began with
  uint32_t *sor_reports = nullptr;
  uint32_t sor_epoch = 0;           // sweeps reported in sor_reports so far
  bool sor_ready = false;           // the loop's buffers are there and sor_reports is cleared
  ufe_path_counts paths{};
  int32_t *d_place = nullptr;       // 0: SOR row; k: edge point k - 1; -k: corner k - 1
  uint8_t *d_skip = nullptr;        // SOR rows prescribed by the grounding-line flux
  bool gl_active = false;
  int64_t *d_chunk_ptr = nullptr;
  int32_t *d_chunk_w = nullptr, *d_col = nullptr;
  uint8_t *d_deg = nullptr;
  double *d_cNx = nullptr, *d_cNy = nullptr;
  double2 *d_cU = nullptr;
  double *d_hNx = nullptr, *d_hNy = nullptr, *d_hNxx = nullptr, *d_hNyy = nullptr;
  double *d_Sxx = nullptr, *d_Sxy = nullptr, *d_Syy = nullptr;
  int colour_start[6] = {0, 0, 0, 0, 0, 0};
  int colour_active[5] = {0, 0, 0, 0, 0};
  // Neumann lists (colour-order indices)
  int32_t *d_neu_row = nullptr, *d_neu_ptr = nullptr, *d_neu_col = nullptr;
  int32_t *d_cor_row = nullptr, *d_cor_ptr = nullptr, *d_cor_col = nullptr;
  int n_neu = 0, n_cor = 0;
  // transposed operator (adjoint): slot coefficients of row q in its neighbours'
  // equations, and the reverse edge-average lists
  double2 *d_cUT = nullptr;
  double *d_cNxT = nullptr, *d_cNyT = nullptr;
  int32_t *d_rev_tgt = nullptr, *d_rev_ptr = nullptr, *d_rev_src = nullptr, *d_rev_cnt = nullptr;
  int n_rev = 0;
  // Aa Neumann for the Aa operator: uses the Aa mesh directly
  // fields
  std::vector<void *> field_ptr;    // per field id (nullptr for pair members)
  double2 *d_pair[3] = {nullptr, nullptr, nullptr};   // W, EV, RHS
  // scratch
  double *d_part = nullptr;         // block partial sums
  int n_part = 0;
  double *d_scalar = nullptr;       // small device scalars
  double *noalloc_scratch = nullptr;   // this device's copy of `scratch` (ufe_ssa_sor_solve_noalloc)
  double *d_tmp[4] = {nullptr, nullptr, nullptr, nullptr};   // nA-sized temporaries
  double *d_ViSMB = nullptr;
  unsigned long long *d_count = nullptr;
  SorFlags *d_flags = nullptr;
  // FP32 copies for the mixed-precision sweeps
  float2 *d_cU32 = nullptr, *d_EV32 = nullptr, *d_R32 = nullptr, *d_D32 = nullptr;
  float *d_Sxy32 = nullptr;
  // Krylov work space (allocated on first use)
  int kry_m = 0;
  bool kry_f32 = true;
  void *kry_V = nullptr, *kry_Z = nullptr, *kry_w = nullptr, *kry_x = nullptr;
  double2 *kry_R64 = nullptr;
  double *bic_S = nullptr;          // BiCGStab scalars on the device
  double *kry_part = nullptr, *kry_H1 = nullptr, *kry_H2 = nullptr, *kry_Hs = nullptr, *kry_y = nullptr,
         *kry_nrm = nullptr;
  double *kry_g = nullptr;          // copies of d_scalar[0..2], after kry_Hs in the same block as kry_H1
  double *h_kry = nullptr;          // pinned host mirror of that block, then the least-squares solution
  // algorithmic bytes per colour (SOR rows only)
  double bytes64[5] = {0, 0, 0, 0, 0}, bytes32[5] = {0, 0, 0, 0, 0};
  double degsum = 0.0;
  // live kernel profile
  bool prof = false;
  int64_t prof_count = 0;
  std::vector<hipEvent_t> ev_pool;
  struct Pending { hipEvent_t a, b; double bytes; int64_t rows; };
  std::vector<Pending> pending;
  ufe_kernel_profile prof_acc{};
  // adjoint work space and Picard checkpoints (allocated on first use)
  int adj_m = 0, adj_K = 0, adj_every = 1, adj_nck = 0;
  bool adj_ready = false;
  double2 *adj_V = nullptr, *adj_Z = nullptr, *adj_w = nullptr, *adj_r = nullptr, *adj_g = nullptr,
          *adj_lam = nullptr, *adj_ubar = nullptr, *adj_uK = nullptr, *adj_pbar = nullptr;
  bool adj_gl = false;               // the forward held the grounding-line rows at the GL-flux velocities
  double *adj_gs = nullptr, *adj_gtau = nullptr, *adj_gA = nullptr, *adj_H1 = nullptr, *adj_Hs = nullptr,
         *adj_y = nullptr, *adj_nrm = nullptr;
  std::vector<double2 *> adj_ck;    // stored iterates u_0, u_c, u_2c, ...
  std::vector<double2 *> adj_seg;   // recomputed iterates of one segment
  ufe_linsolve_opts adj_lin{};
  // batch: the uploaded mesh is a union of independent member meshes (Aa
  // vertices and Ac points in member-major blocks); declared before upload
  std::vector<int32_t> b_nV, b_nAc;  // per member (host, kept across uploads)
  int nb = 0;                        // members of the uploaded mesh (0: single mesh)
  uint16_t *d_mid = nullptr;         // member of each colour-order row
  int n_chunk = 0;                   // SOR-row chunks, each inside one member
  int32_t *d_ch_start = nullptr, *d_ch_count = nullptr, *d_ch_member = nullptr, *d_mch_ptr = nullptr;
  std::vector<int32_t> h_mch_ptr;
  std::vector<int64_t> b_rows;       // SOR rows per member
  // batch Krylov work space and the captured cycle
  int bk_m = 0, bk_ks = 0, bk_prec = -1, bk_bs = 0, bk_sched = -1, bk_loads = -1;
  int bk_key = 0;                   // precision and preconditioner of the captured cycle
  double bk_omega = 0.0;
  void *bk_V = nullptr, *bk_Z = nullptr, *bk_w = nullptr, *bk_x = nullptr, *bk_R = nullptr;
  double *bk_part = nullptr, *bk_H = nullptr, *bk_Hs = nullptr, *bk_y = nullptr, *bk_nrm = nullptr,
         *bk_scale = nullptr, *bk_rel = nullptr, *h_bk_rel = nullptr;
  double bk_tol = 0.0;
  hipGraphExec_t bk_graph = nullptr;
  // autotuned SOR schedule of the batch: threads per block and block order
  int tune_bs = 256, tune_sched = 0, tune_loads = 0;
  bool repeat_turn = false;          // Krylov preconditioner: repeat the turn colour (full sweeps)
  bool neumann_last = true;          // Krylov preconditioner: Neumann update after the last sweep only
  SorFlags *h_flags = nullptr;      // pinned
  double *h_scalar = nullptr;       // pinned
  std::vector<void *> allocs;       // everything to free with the mesh
  // aggregation multigrid preconditioner (built on first use per mesh)
  std::vector<AmgLevel> amg;        // [0] unused (the fine level), coarse levels from 1
  bool amg_ready = false, amg_direct = false, pc_amg = false;
  int amg_nu = 2;                   // smoothing sweeps before and after the coarse correction
  int amg_kfold_max = 0;            // most K-step partials whose step-1 finish a fused cycle folds in
  double *amg_inv = nullptr;
  float2 *amg_y = nullptr;          // fine-level residual v - A z of the restriction
  struct SorGraph {                    // a batch of reference FP64 sweeps, captured
    hipGraphExec_t exec = nullptr;
    int nb = 0, max_sweeps = 0;
    double omega = 0.0, tol = 0.0;
    const uint8_t *skip = nullptr;
  };
  SorGraph sor_graph[8];
  hipGraphExec_t amg_graph = nullptr;   // the coarse levels of one application, captured
  int amg_graph_nu = 0;
  bool amg_T = false;               // cycle the transposed hierarchy (adjoint solves)
  hipGraphExec_t amg_graph_T = nullptr;
  int amg_graph_T_nu = 0;
  double2 *amg_y64 = nullptr;       // FP64 fine-level A z (adjoint)
  double2 *amg_zt64 = nullptr;      // fine vector between the transposed smoothings (patches)
  int fold_max = FOLD_MAX;          // edge points and corners up to which one launch folds (UFE_FOLD_MAX)
  bool cor_apart = false;           // no two corners average the same point, none another corner
  float2 *amg_v32 = nullptr, *amg_z32 = nullptr;   // FP32 copies around an FP64 Krylov method
  float2 *amg_zt = nullptr, *amg_zu = nullptr;     // fine vector between the smoothings (patches)
  double amg_setup_seconds = 0.0;
  int amg_tail_l0 = 0;              // first level solved by k_amg_tail (0: none)
  size_t amg_tail_lds = 0;          // dynamic LDS k_amg_tail may take, bytes
  uint4 *amg_tail_imgA = nullptr, *amg_tail_imgAT = nullptr, *amg_tail_imgB = nullptr;   // staged images
  int amg_tail_wA = 0, amg_tail_wB = 0;                   // their lengths, 16-byte words
  int amg_tail_offA[AMG_TAIL_LEVELS] = {}, amg_tail_offB[AMG_TAIL_LEVELS] = {};
};

#define HIPCHK(ctx, x)                                                            \
  do {                                                                             \
    hipError_t e_ = (x);                                                           \
    if (e_ != hipSuccess) {                                                        \
      (ctx)->err = std::string(#x) + ": " + hipGetErrorString(e_);                \
      return UFE_HIP_ERROR;                                                        \
    }                                                                              \
  } while (0)

#define LAUNCHCHK(ctx)                                                            \
  do {                                                                             \
    hipError_t e_ = hipGetLastError();                                             \
    if (e_ != hipSuccess) {                                                        \
      (ctx)->err = std::string("kernel launch: ") + hipGetErrorString(e_);        \
      return UFE_HIP_ERROR;                                                        \
    }                                                                              \
  } while (0)

// Hilbert-curve index of a point on a 2^16 x 2^16 grid
static uint64_t hilbert_index(uint32_t x, uint32_t y) {
  uint64_t d = 0;
  for (uint32_t s = 1u << 15; s > 0; s >>= 1) {
    const uint32_t rx = (x & s) > 0, ry = (y & s) > 0;
    d += (uint64_t)s * s * ((3 * rx) ^ ry);
    if (ry == 0) {
      if (rx == 1) {
        x = s - 1 - x;
        y = s - 1 - y;
      }
      std::swap(x, y);
    }
  }
  return d;
}

static inline int nblk(int64_t n, int b = BLOCK) { return (int)((n + b - 1) / b); }
// launches per timed sample: odd and no multiple of five, so that the sample goes
// through both smoothings of an application and all colours
constexpr int PROF_EVERY = 7;
// grid for XCD-major kernels: a multiple of the 8 XCDs
static inline int xcd_grid(int64_t n) { return (nblk(n) + 7) / 8 * 8; }
// grid of a layered kernel: points, groups of G layers, fields
static inline dim3 layer_grid(int64_t n, int nz, int G, int fields = 1) {
  return dim3(xcd_grid(n), std::min((nz + G - 1) / G, 65535), fields);
}
// a layered kernel's launch f(width, grid) with the width for n points
template <typename F>
static inline void layered(int64_t n, int nz, int fields, F f) {
  if (nz <= 2 || n * nz <= LAYER_VALUES) f(std::integral_constant<int, 1>{}, layer_grid(n, nz, 1, fields));
  else f(std::integral_constant<int, LAYERS>{}, layer_grid(n, nz, LAYERS, fields));
}

template <typename T>
static int dalloc(ufe_ctx *ctx, T **p, size_t n) {
  *p = nullptr;
  if (n == 0) n = 1;
  HIPCHK(ctx, hipMalloc((void **)p, n * sizeof(T)));
  ctx->allocs.push_back((void *)*p);
  return UFE_OK;
}
template <typename T>
static int dupload(ufe_ctx *ctx, T **p, const T *h, size_t n) {
  int r = dalloc(ctx, p, n);
  if (r) return r;
  if (n) HIPCHK(ctx, hipMemcpyAsync(*p, h, n * sizeof(T), hipMemcpyHostToDevice, ctx->stream));
  return UFE_OK;
}

static void free_mesh(ufe_ctx *ctx) {
  (void)hipStreamSynchronize(ctx->stream);
  for (void *p : ctx->allocs) (void)hipFree(p);
  ctx->allocs.clear();
  ctx->field_ptr.clear();
  ctx->have_mesh = false;
  ctx->d_Tri = ctx->d_niTri = ctx->d_iTri = ctx->d_icount = nullptr;
  ctx->d_NxTri = ctx->d_NyTri = ctx->d_R = ctx->d_crit = nullptr;
  ctx->rm_ready = false;
  ctx->rm_nVs = ctx->rm_nVd = ctx->rm_n = 0;
  if (ctx->rm_work) (void)hipFree(ctx->rm_work);
  ctx->rm_work = nullptr;
  ctx->rm_work_len = 0;
  ctx->d_rm_nn = ctx->d_rm_tvi = ctx->d_rm_st = ctx->d_rm_en = ctx->d_rm_vi = nullptr;
  ctx->d_rm_tw = ctx->d_rm_w0 = ctx->d_rm_w1x = ctx->d_rm_w1y = nullptr;
  // work spaces live in allocs too: forget them with the mesh
  ctx->kry_m = 0;
  ctx->kry_V = ctx->kry_Z = ctx->kry_w = ctx->kry_x = nullptr;
  ctx->kry_R64 = nullptr;
  ctx->bic_S = nullptr;
  ctx->kry_part = ctx->kry_H1 = ctx->kry_H2 = ctx->kry_Hs = ctx->kry_y = ctx->kry_nrm = ctx->kry_g = nullptr;
  ctx->adj_m = ctx->adj_K = ctx->adj_nck = 0;
  ctx->adj_ready = false;
  ctx->adj_V = ctx->adj_Z = ctx->adj_w = ctx->adj_r = ctx->adj_g = ctx->adj_lam = ctx->adj_ubar = ctx->adj_uK =
      ctx->adj_pbar = nullptr;
  ctx->adj_gl = false;
  ctx->adj_gs = ctx->adj_gtau = ctx->adj_gA = ctx->adj_H1 = ctx->adj_Hs = ctx->adj_y = ctx->adj_nrm = nullptr;
  ctx->adj_ck.clear();
  ctx->adj_seg.clear();
  ctx->nb = 0;
  ctx->d_mid = nullptr;
  ctx->n_chunk = 0;
  ctx->d_ch_start = ctx->d_ch_count = ctx->d_ch_member = ctx->d_mch_ptr = nullptr;
  ctx->h_mch_ptr.clear();
  ctx->b_rows.clear();
  ctx->bk_m = ctx->bk_ks = ctx->bk_bs = ctx->bk_key = 0;
  ctx->bk_prec = ctx->bk_sched = -1;
  ctx->bk_V = ctx->bk_Z = ctx->bk_w = ctx->bk_x = ctx->bk_R = nullptr;
  ctx->bk_part = ctx->bk_H = ctx->bk_Hs = ctx->bk_y = ctx->bk_nrm = ctx->bk_scale = ctx->bk_rel = nullptr;
  if (ctx->bk_graph) (void)hipGraphExecDestroy(ctx->bk_graph);
  ctx->bk_graph = nullptr;
  ctx->amg.clear();
  ctx->amg_ready = ctx->amg_direct = false;
  ctx->amg_inv = nullptr;
  ctx->amg_y = nullptr;
  for (auto &G : ctx->sor_graph) {
    if (G.exec) (void)hipGraphExecDestroy(G.exec);
    G = ufe_ctx::SorGraph{};
  }
  if (ctx->amg_graph) (void)hipGraphExecDestroy(ctx->amg_graph);
  ctx->amg_graph = nullptr;
  ctx->amg_graph_nu = 0;
  if (ctx->amg_graph_T) (void)hipGraphExecDestroy(ctx->amg_graph_T);
  ctx->amg_graph_T = nullptr;
  ctx->amg_graph_T_nu = 0;
  ctx->amg_T = false;
  ctx->amg_y64 = ctx->amg_zt64 = nullptr;
  ctx->cor_apart = false;
  ctx->amg_v32 = ctx->amg_z32 = nullptr;
  for (auto &k : ctx->patch)
    for (PatchSet &S : k) S = PatchSet{};
  ctx->d_place = nullptr;
  ctx->sor_w1 = ctx->sor_start = nullptr;
  ctx->sor_reports = nullptr;
  ctx->sor_ready = false;
  ctx->h_key.clear();
  ctx->h_mid.clear();
  ctx->amg_zt = ctx->amg_zu = nullptr;
}

static size_t grid_len(const ufe_ctx *ctx, int grid) {
  switch (grid) {
    case G_AA: return (size_t)ctx->nV;
    case G_AAZ: return (size_t)ctx->nV * ctx->nZ;
    case G_AAC: return (size_t)ctx->nV * ctx->nCm;
    case G_AC: return (size_t)ctx->nAc;
    case G_ACZ: return (size_t)ctx->nAc * ctx->nZ;
    case G_AAAC: return (size_t)ctx->nA;
  }
  return 0;
}

static double *F(ufe_ctx *ctx, const char *name) {
  return (double *)ctx->field_ptr[field_id(name)];
}
static int32_t *FI(ufe_ctx *ctx, const char *name) {
  return (int32_t *)ctx->field_ptr[field_id(name)];
}

static TriMesh tri_mesh(ufe_ctx *c) {
  TriMesh t;
  t.nV = c->nV;
  t.nTri = c->nTri;
  t.V = c->d_V;
  t.Tri = c->d_Tri;
  t.niTri = c->d_niTri;
  t.iTri = c->d_iTri;
  t.NxTri = c->d_NxTri;
  t.NyTri = c->d_NyTri;
  t.R = c->d_R;
  return t;
}

static AaMesh aa_mesh(ufe_ctx *c) {
  AaMesh m;
  m.nV = c->nV;
  m.nCm = c->nCm;
  m.nC = c->d_nC;
  m.C = c->d_C;
  m.edge = c->d_edge;
  m.iAci = c->d_iAci;
  m.Crev = c->d_Crev;
  m.Nx = c->d_Nx;
  m.Ny = c->d_Ny;
  m.Nxx = c->d_Nxx;
  m.Nxy = c->d_Nxy;
  m.Nyy = c->d_Nyy;
  m.A = c->d_A;
  m.Cw = c->d_Cw;
  return m;
}
static AcMesh ac_mesh(ufe_ctx *c) {
  AcMesh m;
  m.nAc = c->nAc;
  m.nV = c->nV;
  m.Aci = c->d_Aci;
  m.Nx = c->d_NxAc;
  m.Ny = c->d_NyAc;
  m.No = c->d_NoAc;
  m.Np = c->d_NpAc;
  m.edge = c->d_edgeAc;
  m.slot_i = c->d_slot_i;
  m.slot_j = c->d_slot_j;
  m.V = c->d_V;
  return m;
}
static AaAcMesh aaac_mesh(ufe_ctx *c) {
  AaAcMesh m;
  m.nA = c->nA;
  m.nV = c->nV;
  m.perm = c->d_perm;
  m.chunk_ptr = c->d_chunk_ptr;
  m.chunk_w = c->d_chunk_w;
  m.deg = c->d_deg;
  m.col = c->d_col;
  m.cNx = c->d_cNx;
  m.cNy = c->d_cNy;
  m.cU = c->d_cU;
  m.hNx = c->d_hNx;
  m.hNy = c->d_hNy;
  m.hNxx = c->d_hNxx;
  m.hNyy = c->d_hNyy;
  m.Sxx = c->d_Sxx;
  m.Sxy = c->d_Sxy;
  m.Syy = c->d_Syy;
  return m;
}
static SSAFields ssa_fields(ufe_ctx *c) {
  SSAFields f;
  f.Hi = F(c, "Hi_AaAc");
  f.Hb = F(c, "Hb_AaAc");
  f.SL = F(c, "SL_AaAc");
  f.dsx = F(c, "dHs_dx_shelf_AaAc");
  f.dsy = F(c, "dHs_dy_shelf_AaAc");
  f.Aflow = F(c, "A_flow_mean_AaAc");
  f.ux = F(c, "dU_SSA_dx_AaAc");
  f.uy = F(c, "dU_SSA_dy_AaAc");
  f.vx = F(c, "dV_SSA_dx_AaAc");
  f.vy = F(c, "dV_SSA_dy_AaAc");
  f.eta = F(c, "eta_AaAc");
  f.N = F(c, "N_AaAc");
  f.Nprev = F(c, "N_AaAc_prev");
  f.S = F(c, "S_AaAc");
  f.phi = F(c, "phi_fric_AaAc");
  f.tau = F(c, "tau_c_AaAc");
  f.tau_ovr = F(c, "tau_c_override_AaAc");
  f.W = c->d_pair[0];
  f.EV = c->d_pair[1];
  f.RHS = c->d_pair[2];
  return f;
}

static ufe_params default_params() {
  ufe_params p{};
  const double z[15] = {0.00, 0.10, 0.20, 0.30, 0.40, 0.50, 0.60, 0.70,
                        0.80, 0.90, 0.925, 0.95, 0.975, 0.99, 1.00};
  p.nZ = 15;
  for (int k = 0; k < 15; k++) p.zeta[k] = z[k];
  p.m_enh_sia = 5.0;
  p.m_enh_ssa = 0.7;
  p.SSA_RN_tol = 1e-5;
  p.SSA_max_outer_loops = 50;
  p.SSA_max_residual_UV = 2.5;
  p.SSA_SOR_omega = 1.2;
  p.SSA_max_inner_loops = 10000;
  p.zero_Hi_at_edges = 1;
  p.precision = UFE_FP64;
  return p;
}

// ---------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------
// ---- scratch of the allocation-free SOR solve -------------------------------
// ufe_ssa_sor_solve_noalloc keeps the FP64 residual's block partial sums and
// its result here instead of in context buffers.  Each GPU holds its own copy
// for the life of the process; host code reaches it only through the address
// hipGetSymbolAddress gives for that device (the array's name is a host-side
// stand-in, not a device address).
constexpr int NOALLOC_MAX_ROWS = 1 << 23;                      // SOR rows (nVAaAc) at most
constexpr int NOALLOC_PARTS = NOALLOC_MAX_ROWS / BLOCK + 8;    // residual blocks: one extra per colour
constexpr int NOALLOC_DOUBLES = 2 * NOALLOC_PARTS + 8;         // partial pairs, then the result
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];
constexpr int NOALLOC_DEVICES = 64;
static double *g_scratch_addr[NOALLOC_DEVICES];
static std::mutex g_scratch_mu;

// Device address of `scratch` on `device`, which must be current; looked up
// once per device.
static int noalloc_scratch_setup(int device, double **out) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (device < 0 || device >= NOALLOC_DEVICES) return UFE_BAD_INPUT;
  if (!g_scratch_addr[device]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      (void)hipGetLastError();
      return UFE_HIP_ERROR;
    }
    g_scratch_addr[device] = static_cast<double *>(p);
  }
  *out = g_scratch_addr[device];
  return UFE_OK;
}

// An exception from host code (memory or threads exhausted) ends the entry
// point it reached with UFE_HOST_ERROR; none leaves through the C interface.
static int host_failure(ufe_ctx *ctx, const char *what) {
  if (ctx) ctx->err = std::string("host failure: ") + (what ? what : "");
  return UFE_HOST_ERROR;
}

extern "C" {

int ufe_version(void) { return 1; }

const char *ufe_last_error(ufe_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int ufe_ctx_create(int device, ufe_ctx **out) try {
  if (!out) return UFE_BAD_INPUT;
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= device || device < 0) return UFE_HIP_ERROR;
  ufe_ctx *ctx = new ufe_ctx();
  ctx->device = device;
  ctx->params = default_params();
  if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess ||
      hipHostMalloc((void **)&ctx->h_flags, sizeof(SorFlags), hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void **)&ctx->h_scalar, 8 * sizeof(double), hipHostMallocDefault) != hipSuccess) {
    delete ctx;
    return UFE_HIP_ERROR;
  }
  // the allocation-free solve's scratch on this device (left null on failure:
  // that entry point then refuses with UFE_HIP_ERROR, the others are unaffected)
  if (noalloc_scratch_setup(device, &ctx->noalloc_scratch) != UFE_OK) ctx->noalloc_scratch = nullptr;
  *out = ctx;
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(nullptr, e.what());
} catch (...) {
  return host_failure(nullptr, "unknown exception");
}

int ufe_ctx_destroy(ufe_ctx *ctx) {
  if (!ctx) return UFE_OK;
  (void)hipSetDevice(ctx->device);
  free_mesh(ctx);
  for (auto &p : ctx->pending) {
    (void)hipEventDestroy(p.a);
    (void)hipEventDestroy(p.b);
  }
  for (auto e : ctx->ev_pool) (void)hipEventDestroy(e);
  if (ctx->h_flags) (void)hipHostFree(ctx->h_flags);
  if (ctx->h_scalar) (void)hipHostFree(ctx->h_scalar);
  if (ctx->h_kry) (void)hipHostFree(ctx->h_kry);
  if (ctx->h_bk_rel) (void)hipHostFree(ctx->h_bk_rel);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
  return UFE_OK;
}

int ufe_set_params(ufe_ctx *ctx, const ufe_params *p) {
  if (!ctx || !p) return UFE_BAD_INPUT;
  if (p->nZ < 2 || p->nZ > MAX_NZ) {
    ctx->err = "nZ out of range";
    return UFE_BAD_INPUT;
  }
  if (ctx->have_mesh && p->nZ != ctx->nZ) {
    ctx->err = "nZ cannot change after mesh upload";
    return UFE_BAD_INPUT;
  }
  if (p->precision != UFE_FP64 && p->precision != UFE_MIXED && p->precision != UFE_FP64_KRYLOV) {
    ctx->err = "precision must be UFE_FP64, UFE_MIXED or UFE_FP64_KRYLOV";
    return UFE_BAD_INPUT;
  }
  if (p->SSA_gmres_restart > 64) {
    ctx->err = "SSA_gmres_restart must be at most 64";
    return UFE_BAD_INPUT;
  }
  if (p->SSA_precond_type != UFE_PRECOND_SOR &&
      !(p->SSA_precond_type == UFE_PRECOND_MULTIGRID && p->precision != UFE_FP64)) {
    ctx->err = "SSA_precond_type must be UFE_PRECOND_SOR, or UFE_PRECOND_MULTIGRID with UFE_MIXED or UFE_FP64_KRYLOV";
    return UFE_BAD_INPUT;
  }
  ctx->params = *p;
  ctx->nZ = p->nZ;
  return UFE_OK;
}

int ufe_field_count(void) { return NFIELDS; }
const char *ufe_field_name(int id) { return (id >= 0 && id < NFIELDS) ? FIELDS[id].name : nullptr; }
int ufe_field_id(const char *name) { return name ? field_id(name) : -1; }
int ufe_field_info(int id, int32_t *grid, int32_t *dtype) {
  if (id < 0 || id >= NFIELDS) return UFE_BAD_INPUT;
  if (grid) *grid = FIELDS[id].grid;
  if (dtype) *dtype = FIELDS[id].dtype;
  return UFE_OK;
}

int ufe_synchronize(ufe_ctx *ctx) {
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}
int ufe_device_alloc(ufe_ctx *ctx, size_t bytes, void **dev) {
  HIPCHK(ctx, hipMalloc(dev, bytes));
  return UFE_OK;
}
int ufe_device_free(ufe_ctx *ctx, void *dev) {
  HIPCHK(ctx, hipFree(dev));
  return UFE_OK;
}
int ufe_memcpy_h2d(ufe_ctx *ctx, void *dev, const void *host, size_t bytes) {
  HIPCHK(ctx, hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}
int ufe_memcpy_d2h(ufe_ctx *ctx, void *host, const void *dev, size_t bytes) {
  HIPCHK(ctx, hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

int ufe_mesh_sizes(ufe_ctx *ctx, int32_t *out4) {
  if (!ctx || !ctx->have_mesh || !out4) return UFE_BAD_INPUT;
  out4[0] = ctx->nV;
  out4[1] = ctx->nAc;
  out4[2] = ctx->nA;
  out4[3] = ctx->nCm;
  return UFE_OK;
}

// ---- mesh build ------------------------------------------------------------
static int check_primary(ufe_ctx *ctx, const ufe_mesh_desc *m) {
  if (!m || m->nV < 5 || m->nTri < 4 || m->nC_mem < 3 || m->nC_mem > NF_MAX || !m->V || !m->nC ||
      !m->C || !m->niTri || !m->iTri || !m->edge_index || !m->Tri) {
    ctx->err = "mesh descriptor incomplete or nC_mem outside [3,16]";
    return UFE_BAD_INPUT;
  }
  int64_t s = 0;
  for (int v = 0; v < m->nV; v++) {
    if (m->nC[v] < 2 || m->nC[v] > m->nC_mem) {
      ctx->err = "nC out of range";
      return UFE_BAD_INPUT;
    }
    s += m->nC[v];
  }
  if (s % 2 || s / 2 != m->nAc) {
    ctx->err = "nAc must equal (sum of nC)/2";
    return UFE_BAD_INPUT;
  }
  for (int v = 0; v < m->nV; v++)
    for (int c = 0; c < m->nC[v]; c++) {
      const int j = m->C[(int64_t)c * m->nV + v];
      if (j < 1 || j > m->nV) {
        ctx->err = "C holds an index outside 1..nV";
        return UFE_BAD_INPUT;
      }
    }
  // triangles: the upwind derivatives and triangle neighbour functions index through them
  for (int v = 0; v < m->nV; v++) {
    if (m->niTri[v] < 1 || m->niTri[v] > m->nC_mem) {
      ctx->err = "niTri out of range";
      return UFE_BAD_INPUT;
    }
    for (int c = 0; c < m->niTri[v]; c++) {
      const int t = m->iTri[(int64_t)c * m->nV + v];
      if (t < 1 || t > m->nTri) {
        ctx->err = "iTri holds an index outside 1..nTri";
        return UFE_BAD_INPUT;
      }
    }
  }
  for (int64_t k = 0; k < 3 * (int64_t)m->nTri; k++)
    if (m->Tri[k] < 1 || m->Tri[k] > m->nV) {
      ctx->err = "Tri holds an index outside 1..nV";
      return UFE_BAD_INPUT;
    }
  return UFE_OK;
}

static int gpu_neighbour_functions(ufe_ctx *ctx, int np, int nCm, const double *V, const int32_t *nc,
                                   const int32_t *cl, int split, const int32_t *edge_aa, int nV,
                                   const int32_t *edge_ac, int nAc, double *Nx, double *Ny,
                                   double *Nxx, double *Nxy, double *Nyy) {
  double *dV, *dN[5];
  int32_t *dnc, *dcl, *dea, *dec;
  const size_t w = (size_t)np * (nCm + 1);
  HIPCHK(ctx, hipMalloc((void **)&dV, sizeof(double) * 2 * np));
  HIPCHK(ctx, hipMalloc((void **)&dnc, sizeof(int32_t) * np));
  HIPCHK(ctx, hipMalloc((void **)&dcl, sizeof(int32_t) * (size_t)np * nCm));
  HIPCHK(ctx, hipMalloc((void **)&dea, sizeof(int32_t) * std::max(nV, 1)));
  HIPCHK(ctx, hipMalloc((void **)&dec, sizeof(int32_t) * std::max(nAc, 1)));
  for (int k = 0; k < 5; k++) HIPCHK(ctx, hipMalloc((void **)&dN[k], sizeof(double) * w));
  HIPCHK(ctx, hipMemcpyAsync(dV, V, sizeof(double) * 2 * np, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(ctx, hipMemcpyAsync(dnc, nc, sizeof(int32_t) * np, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(ctx, hipMemcpyAsync(dcl, cl, sizeof(int32_t) * (size_t)np * nCm, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(ctx, hipMemcpyAsync(dea, edge_aa, sizeof(int32_t) * nV, hipMemcpyHostToDevice, ctx->stream));
  if (nAc) HIPCHK(ctx, hipMemcpyAsync(dec, edge_ac, sizeof(int32_t) * nAc, hipMemcpyHostToDevice, ctx->stream));
  k_neighbour_functions<<<nblk(np, 128), 128, 0, ctx->stream>>>(np, nCm, dV, dnc, dcl, split, dea, dec,
                                                              dN[0], dN[1], dN[2], dN[3], dN[4]);
  LAUNCHCHK(ctx);
  double *out[5] = {Nx, Ny, Nxx, Nxy, Nyy};
  for (int k = 0; k < 5; k++)
    HIPCHK(ctx, hipMemcpyAsync(out[k], dN[k], sizeof(double) * w, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  (void)hipFree(dV);
  (void)hipFree(dnc);
  (void)hipFree(dcl);
  (void)hipFree(dea);
  (void)hipFree(dec);
  for (int k = 0; k < 5; k++) (void)hipFree(dN[k]);
  return UFE_OK;
}

int ufe_mesh_build(ufe_ctx *ctx, ufe_mesh_desc *m) try {
  if (!ctx) return UFE_BAD_INPUT;
  int r = check_primary(ctx, m);
  if (r) return r;
  if (!m->iAci || !m->Aci || !m->VAc || !m->Nx_Ac || !m->Ny_Ac || !m->No_Ac || !m->Np_Ac ||
      !m->edge_index_Ac || !m->VAaAc || !m->nCAaAc || !m->CAaAc || !m->Nx_AaAc || !m->Ny_AaAc ||
      !m->Nxx_AaAc || !m->Nxy_AaAc || !m->Nyy_AaAc || !m->Nx || !m->Ny || !m->Nxx || !m->Nxy ||
      !m->Nyy || !m->colour || !m->colour_vi) {
    ctx->err = "mesh descriptor lacks secondary output arrays";
    return UFE_BAD_INPUT;
  }
  HIPCHK(ctx, hipSetDevice(ctx->device));
  if ((r = build_Ac_mesh(m, ctx->err))) return r;
  if ((r = build_AaAc_connectivity(m, ctx->err))) return r;
  const int nV = m->nV, nA = m->nV + m->nAc;
  // neighbour functions of the AaAc points (src/mesh_ArakawaC_module.f90:511-537)
  if ((r = gpu_neighbour_functions(ctx, nA, m->nC_mem, m->VAaAc, m->nCAaAc, m->CAaAc, nV,
                                   m->edge_index, nV, m->edge_index_Ac, m->nAc, m->Nx_AaAc,
                                   m->Ny_AaAc, m->Nxx_AaAc, m->Nxy_AaAc, m->Nyy_AaAc)))
    return r;
  // and of the Aa vertices (src/mesh_derivatives_module.f90:51-70)
  if ((r = gpu_neighbour_functions(ctx, nV, m->nC_mem, m->V, m->nC, m->C, nV, m->edge_index, nV,
                                   m->edge_index_Ac, 0, m->Nx, m->Ny, m->Nxx, m->Nxy, m->Nyy)))
    return r;
  return five_colouring(m, ctx->err);
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

// ---- primary-mesh geometry ---------------------------------------------------
namespace {
// Device scratch of one call, released on every return path.
struct ScratchDev {
  std::vector<void *> ptrs;
  ~ScratchDev() {
    for (void *p : ptrs) (void)hipFree(p);
  }
  hipError_t alloc(void **p, size_t bytes) {
    *p = nullptr;
    hipError_t e = hipMalloc(p, std::max<size_t>(bytes, 8));
    if (e == hipSuccess) ptrs.push_back(*p);
    return e;
  }
};
}  // namespace

static int check_geometry(ufe_ctx *ctx, const ufe_mesh_geometry_desc *g) {
  auto bad = [&](const char *msg) {
    ctx->err = std::string("ufe_mesh_geometry: ") + msg;
    return UFE_BAD_INPUT;
  };
  if (!g || !g->V || !g->nC || !g->C || !g->niTri || !g->iTri || !g->edge_index || !g->Tri ||
      !g->Tri_edge_index || !g->Tricc)
    return bad("descriptor incomplete");
  if (g->nV < 3 || g->nTri < 1 || g->nC_mem < 3 || g->nC_mem > 64) return bad("sizes out of range");
  if (!(g->xmax > g->xmin) || !(g->ymax > g->ymin) || !(g->tol_dist >= 0.0)) return bad("domain bounds");
  const int64_t lv = g->nV, lt = g->nTri;
  for (int v = 0; v < g->nV; v++) {
    if (g->nC[v] < 0 || g->nC[v] > g->nC_mem) return bad("nC out of range");
    if (g->niTri[v] < 0 || g->niTri[v] > g->nC_mem) return bad("niTri out of range");
    for (int c = 0; c < g->nC[v]; c++) {
      const int j = g->C[c * lv + v];
      if (j < 1 || j > g->nV) return bad("C holds an index outside 1..nV");
    }
    for (int c = 0; c < g->niTri[v]; c++) {
      const int t = g->iTri[c * lv + v];
      if (t < 1 || t > g->nTri) return bad("iTri holds an index outside 1..nTri");
    }
  }
  for (int64_t k = 0; k < 3 * lt; k++)
    if (g->Tri[k] < 1 || g->Tri[k] > g->nV) return bad("Tri holds an index outside 1..nV");
  return UFE_OK;
}

int ufe_mesh_geometry(ufe_ctx *ctx, ufe_mesh_geometry_desc *g, ufe_mesh_geometry_stats *st) try {
  if (!ctx) return UFE_BAD_INPUT;
  int r = check_geometry(ctx, g);
  if (r) return r;
  HIPCHK(ctx, hipSetDevice(ctx->device));
  const size_t nV = g->nV, nT = g->nTri, nCm = g->nC_mem;
  ScratchDev s;
  GeomMesh m;
  m.nV = g->nV;
  m.nTri = g->nTri;
  m.nCm = g->nC_mem;
  m.xmin = g->xmin;
  m.xmax = g->xmax;
  m.ymin = g->ymin;
  m.ymax = g->ymax;
  m.tol = g->tol_dist;
  double *dV, *dcc, *dA = nullptr, *dCw = nullptr, *dTriA = nullptr, *dR = nullptr;
  int32_t *dnC, *dC, *dniTri, *diTri, *dedge, *dTri, *dtei, *dcount;
  HIPCHK(ctx, s.alloc((void **)&dV, sizeof(*dV) * (2 * nV)));
  HIPCHK(ctx, s.alloc((void **)&dnC, sizeof(*dnC) * (nV)));
  HIPCHK(ctx, s.alloc((void **)&dC, sizeof(*dC) * (nV * nCm)));
  HIPCHK(ctx, s.alloc((void **)&dniTri, sizeof(*dniTri) * (nV)));
  HIPCHK(ctx, s.alloc((void **)&diTri, sizeof(*diTri) * (nV * nCm)));
  HIPCHK(ctx, s.alloc((void **)&dedge, sizeof(*dedge) * (nV)));
  HIPCHK(ctx, s.alloc((void **)&dTri, sizeof(*dTri) * (3 * nT)));
  HIPCHK(ctx, s.alloc((void **)&dtei, sizeof(*dtei) * (nT)));
  HIPCHK(ctx, s.alloc((void **)&dcc, sizeof(*dcc) * (2 * nT)));
  HIPCHK(ctx, s.alloc((void **)&dcount, sizeof(*dcount) * (GEO_NCOUNT)));
  if (g->A) HIPCHK(ctx, s.alloc((void **)&dA, sizeof(*dA) * (nV)));
  if (g->Cw) HIPCHK(ctx, s.alloc((void **)&dCw, sizeof(*dCw) * (nV * nCm)));
  if (g->TriA) HIPCHK(ctx, s.alloc((void **)&dTriA, sizeof(*dTriA) * (nT)));
  if (g->R) HIPCHK(ctx, s.alloc((void **)&dR, sizeof(*dR) * (nV)));
  hipStream_t q = ctx->stream;
  HIPCHK(ctx, hipMemcpyAsync(dV, g->V, sizeof(double) * 2 * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(dnC, g->nC, sizeof(int32_t) * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(dC, g->C, sizeof(int32_t) * nV * nCm, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(dniTri, g->niTri, sizeof(int32_t) * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(diTri, g->iTri, sizeof(int32_t) * nV * nCm, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(dedge, g->edge_index, sizeof(int32_t) * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(dTri, g->Tri, sizeof(int32_t) * 3 * nT, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(dtei, g->Tri_edge_index, sizeof(int32_t) * nT, hipMemcpyHostToDevice, q));
  if (!g->compute_Tricc)
    HIPCHK(ctx, hipMemcpyAsync(dcc, g->Tricc, sizeof(double) * 2 * nT, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemsetAsync(dcount, 0, sizeof(int32_t) * GEO_NCOUNT, q));
  m.V = dV;
  m.nC = dnC;
  m.C = dC;
  m.niTri = dniTri;
  m.iTri = diTri;
  m.edge = dedge;
  m.Tri = dTri;
  m.tei = dtei;
  m.cc = dcc;
  if (g->compute_Tricc) k_geo_tricc<<<nblk(g->nTri), BLOCK, 0, q>>>(m, dcount);
  if (dTriA) k_geo_tri_area<<<nblk(g->nTri), BLOCK, 0, q>>>(m, dTriA);
  if (dA) k_geo_voronoi_area<<<nblk(g->nV), BLOCK, 0, q>>>(m, dA, dcount);
  if (dCw) k_geo_conn_width<<<nblk(g->nV), BLOCK, 0, q>>>(m, dCw, dcount);
  if (dR) k_geo_resolution<<<nblk(g->nV), BLOCK, 0, q>>>(m, dR);
  LAUNCHCHK(ctx);
  int32_t count[GEO_NCOUNT];
  HIPCHK(ctx, hipMemcpyAsync(count, dcount, sizeof(count), hipMemcpyDeviceToHost, q));
  if (g->compute_Tricc) {
    HIPCHK(ctx, hipMemcpyAsync(g->Tricc, dcc, sizeof(double) * 2 * nT, hipMemcpyDeviceToHost, q));
    HIPCHK(ctx, hipMemcpyAsync(g->Tri, dTri, sizeof(int32_t) * 3 * nT, hipMemcpyDeviceToHost, q));
  }
  if (dA) HIPCHK(ctx, hipMemcpyAsync(g->A, dA, sizeof(double) * nV, hipMemcpyDeviceToHost, q));
  if (dCw) HIPCHK(ctx, hipMemcpyAsync(g->Cw, dCw, sizeof(double) * nV * nCm, hipMemcpyDeviceToHost, q));
  if (dTriA) HIPCHK(ctx, hipMemcpyAsync(g->TriA, dTriA, sizeof(double) * nT, hipMemcpyDeviceToHost, q));
  if (dR) HIPCHK(ctx, hipMemcpyAsync(g->R, dR, sizeof(double) * nV, hipMemcpyDeviceToHost, q));
  HIPCHK(ctx, hipStreamSynchronize(q));
  ufe_mesh_geometry_stats t{};
  t.rotated_triangles = count[GEO_ROTATED];
  t.invalid_circumcentres = count[GEO_INVALID_CC];
  t.voronoi_outside = count[GEO_OUTSIDE] + count[GEO_TOPOLOGY];
  t.connection_failures = count[GEO_CW_FAIL];
  if (g->A) {
    double sum = 0.0;   // SUM(mesh%A), sequential
    for (size_t v = 0; v < nV; v++) sum = sum + g->A[v];
    t.area_error = std::fabs(1.0 - sum / ((g->xmax - g->xmin) * (g->ymax - g->ymin)));
  }
  if (g->R) {
    t.resolution_min = t.resolution_max = g->R[0];
    for (size_t v = 1; v < nV; v++) {
      t.resolution_min = std::min(t.resolution_min, g->R[v]);
      t.resolution_max = std::max(t.resolution_max, g->R[v]);
    }
  }
  if (st) *st = t;
  if (t.invalid_circumcentres) {
    ctx->err = "ufe_mesh_geometry: a triangle does not yield a valid circumcentre";
    return UFE_BAD_INPUT;
  }
  if (t.voronoi_outside) {
    ctx->err = "ufe_mesh_geometry: found Voronoi cell vertices outside of the mesh domain";
    return UFE_BAD_INPUT;
  }
  if (t.connection_failures) {
    ctx->err = "ufe_mesh_geometry: a connection has no shared triangle, or one that is not a boundary triangle";
    return UFE_BAD_INPUT;
  }
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}


// ---- remapping between meshes -------------------------------------------------
namespace {
// Device copy of one primary mesh with its geometry, for the remapping build.
struct GeoDev {
  GeomMesh m{};
  const double *A = nullptr;
};
}  // namespace

static int upload_geo(ufe_ctx *ctx, ScratchDev &s, const ufe_mesh_geometry_desc *g, GeoDev &out) {
  const size_t nV = g->nV, nT = g->nTri, nCm = g->nC_mem;
  double *V, *cc, *A;
  int32_t *nC, *C, *niTri, *iTri, *edge, *Tri, *tei;
  HIPCHK(ctx, s.alloc((void **)&V, sizeof(double) * 2 * nV));
  HIPCHK(ctx, s.alloc((void **)&cc, sizeof(double) * 2 * nT));
  HIPCHK(ctx, s.alloc((void **)&A, sizeof(double) * nV));
  HIPCHK(ctx, s.alloc((void **)&nC, sizeof(int32_t) * nV));
  HIPCHK(ctx, s.alloc((void **)&C, sizeof(int32_t) * nV * nCm));
  HIPCHK(ctx, s.alloc((void **)&niTri, sizeof(int32_t) * nV));
  HIPCHK(ctx, s.alloc((void **)&iTri, sizeof(int32_t) * nV * nCm));
  HIPCHK(ctx, s.alloc((void **)&edge, sizeof(int32_t) * nV));
  HIPCHK(ctx, s.alloc((void **)&Tri, sizeof(int32_t) * 3 * nT));
  HIPCHK(ctx, s.alloc((void **)&tei, sizeof(int32_t) * nT));
  hipStream_t q = ctx->stream;
  HIPCHK(ctx, hipMemcpyAsync(V, g->V, sizeof(double) * 2 * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(cc, g->Tricc, sizeof(double) * 2 * nT, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(A, g->A, sizeof(double) * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(nC, g->nC, sizeof(int32_t) * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(C, g->C, sizeof(int32_t) * nV * nCm, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(niTri, g->niTri, sizeof(int32_t) * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(iTri, g->iTri, sizeof(int32_t) * nV * nCm, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(edge, g->edge_index, sizeof(int32_t) * nV, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(Tri, g->Tri, sizeof(int32_t) * 3 * nT, hipMemcpyHostToDevice, q));
  HIPCHK(ctx, hipMemcpyAsync(tei, g->Tri_edge_index, sizeof(int32_t) * nT, hipMemcpyHostToDevice, q));
  GeomMesh &m = out.m;
  m.nV = g->nV;
  m.nTri = g->nTri;
  m.nCm = g->nC_mem;
  m.xmin = g->xmin;
  m.xmax = g->xmax;
  m.ymin = g->ymin;
  m.ymax = g->ymax;
  m.tol = g->tol_dist;
  m.V = V;
  m.nC = nC;
  m.C = C;
  m.niTri = niTri;
  m.iTri = iTri;
  m.edge = edge;
  m.Tri = Tri;
  m.tei = tei;
  m.cc = cc;
  out.A = A;
  return UFE_OK;
}

static double rm_area_host(const double *a, const double *b, const double *c) {
  return std::fabs((b[0] - a[0]) * (c[1] - a[1]) - (b[1] - a[1]) * (c[0] - a[0])) / 2.0;
}

int ufe_remap_build(ufe_ctx *dst, ufe_ctx *src, const ufe_mesh_geometry_desc *gs, const ufe_mesh_geometry_desc *gd,
                    ufe_remap_stats *st) try {
  if (!dst || !src || !dst->have_mesh || !src->have_mesh) return UFE_BAD_INPUT;
  if (dst->device != src->device) {
    dst->err = "ufe_remap_build: both contexts must use the same device";
    return UFE_BAD_INPUT;
  }
  int r;
  if ((r = check_geometry(dst, gs)) || (r = check_geometry(dst, gd))) return r;
  if (!gs->A || !gd->A || gs->nV != src->nV || gd->nV != dst->nV || gs->nC_mem > 32 || gd->nC_mem > 32) {
    dst->err = "ufe_remap_build: geometry descriptors must hold A and match the two meshes (nC_mem <= 32)";
    return UFE_BAD_INPUT;
  }
  const auto t0 = std::chrono::steady_clock::now();
  HIPCHK(dst, hipSetDevice(dst->device));
  HIPCHK(dst, hipStreamSynchronize(src->stream));
  hipStream_t q = dst->stream;
  const int nVs = gs->nV, nVd = gd->nV;
  ScratchDev s;
  GeoDev S, D;
  if ((r = upload_geo(dst, s, gs, S)) || (r = upload_geo(dst, s, gd, D))) return r;
  double *Ps, *Pd, *GCs;
  int32_t *nPs, *nPd, *cnt, *count;
  HIPCHK(dst, s.alloc((void **)&Ps, sizeof(double) * 2 * RM_MAXP * (size_t)nVs));
  HIPCHK(dst, s.alloc((void **)&Pd, sizeof(double) * 2 * RM_MAXP * (size_t)nVd));
  HIPCHK(dst, s.alloc((void **)&GCs, sizeof(double) * 2 * (size_t)nVs));
  HIPCHK(dst, s.alloc((void **)&nPs, sizeof(int32_t) * nVs));
  HIPCHK(dst, s.alloc((void **)&nPd, sizeof(int32_t) * nVd));
  HIPCHK(dst, s.alloc((void **)&cnt, sizeof(int32_t) * nVd));
  HIPCHK(dst, s.alloc((void **)&count, sizeof(int32_t) * RM_NCOUNT));
  HIPCHK(dst, hipMemsetAsync(count, 0, sizeof(int32_t) * RM_NCOUNT, q));
  k_rm_cells<<<nblk(nVs, 64), 64, 0, q>>>(S.m, S.A, Ps, nPs, GCs, count);
  k_rm_cells<<<nblk(nVd, 64), 64, 0, q>>>(D.m, D.A, Pd, nPd, nullptr, count);
  LAUNCHCHK(dst);
  // bucket grid of the source vertices: about one vertex per cell
  const double Lx = gs->xmax - gs->xmin, Ly = gs->ymax - gs->ymin;
  const double h = std::sqrt(Lx * Ly / std::max(nVs, 1));
  RmGrid G;
  G.nx = std::max(1, (int)std::ceil(Lx / h));
  G.ny = std::max(1, (int)std::ceil(Ly / h));
  G.x0 = gs->xmin;
  G.y0 = gs->ymin;
  G.h = h;
  std::vector<int32_t> gstart((size_t)G.nx * G.ny + 1, 0), gitem(nVs), cell(nVs);
  for (int v = 0; v < nVs; v++) {
    int cx = (int)std::floor((gs->V[v] - G.x0) / h), cy = (int)std::floor((gs->V[nVs + v] - G.y0) / h);
    cx = std::min(std::max(cx, 0), G.nx - 1);
    cy = std::min(std::max(cy, 0), G.ny - 1);
    cell[v] = cy * G.nx + cx;
    gstart[cell[v] + 1]++;
  }
  for (size_t c = 0; c + 1 < gstart.size(); c++) gstart[c + 1] += gstart[c];
  {
    std::vector<int32_t> fillp(gstart.begin(), gstart.end() - 1);
    for (int v = 0; v < nVs; v++) gitem[fillp[cell[v]]++] = v;
  }
  int32_t *dgs, *dgi;
  HIPCHK(dst, s.alloc((void **)&dgs, sizeof(int32_t) * gstart.size()));
  HIPCHK(dst, s.alloc((void **)&dgi, sizeof(int32_t) * std::max(nVs, 1)));
  HIPCHK(dst, hipMemcpyAsync(dgs, gstart.data(), sizeof(int32_t) * gstart.size(), hipMemcpyHostToDevice, q));
  HIPCHK(dst, hipMemcpyAsync(dgi, gitem.data(), sizeof(int32_t) * nVs, hipMemcpyHostToDevice, q));
  G.start = dgs;
  G.item = dgi;
  // persistent arrays of the remapping, freed with the destination mesh
  dst->rm_ready = false;
  if ((r = dalloc(dst, &dst->d_rm_nn, nVd)) || (r = dalloc(dst, &dst->d_rm_tvi, 3 * (size_t)nVd)) ||
      (r = dalloc(dst, &dst->d_rm_tw, 3 * (size_t)nVd)) || (r = dalloc(dst, &dst->d_rm_st, nVd)) ||
      (r = dalloc(dst, &dst->d_rm_en, nVd)))
    return r;
  k_rm_nearest<<<nblk(nVd), BLOCK, 0, q>>>(nVd, D.m.V, G, S.m.V, nVs, dst->d_rm_nn);
  k_rm_trilin<<<nblk(nVd, 64), 64, 0, q>>>(nVd, D.m.V, S.m, dst->d_rm_nn, dst->d_rm_tvi, dst->d_rm_tw, count);
  LAUNCHCHK(dst);
  RmCons R;
  R.nVd = nVd;
  R.Pd = Pd;
  R.Ps = Ps;
  R.nPd = nPd;
  R.nPs = nPs;
  R.Ad = D.A;
  R.GCs = GCs;
  R.edge_d = D.m.edge;
  R.nn = dst->d_rm_nn;
  R.nCs = S.m.nC;
  R.Cs = S.m.C;
  R.nVs = nVs;
  R.xmin = gd->xmin;
  R.xmax = gd->xmax;
  R.ymin = gd->ymin;
  R.ymax = gd->ymax;
  R.tol = gd->tol_dist;
  k_rm_cons<<<nblk(nVd, 64), 64, 0, q>>>(R, 0, nullptr, cnt, nullptr, nullptr, nullptr, nullptr, count);
  LAUNCHCHK(dst);
  std::vector<int32_t> hc(nVd), hst(nVd), hen(nVd);
  HIPCHK(dst, hipMemcpyAsync(hc.data(), cnt, sizeof(int32_t) * nVd, hipMemcpyDeviceToHost, q));
  int32_t hcount[RM_NCOUNT];
  HIPCHK(dst, hipMemcpyAsync(hcount, count, sizeof(hcount), hipMemcpyDeviceToHost, q));
  HIPCHK(dst, hipStreamSynchronize(q));
  if (hcount[RM_OVERFLOW]) {
    dst->err = "ufe_remap_build: a cell polygon or overlap list exceeds its capacity";
    return UFE_BAD_INPUT;
  }
  int64_t tot = 0;
  for (int v = 0; v < nVd; v++) {
    hst[v] = (int32_t)tot;
    tot += hc[v];
    hen[v] = (int32_t)tot;
  }
  if (tot > INT32_MAX) {
    dst->err = "ufe_remap_build: too many remapping entries";
    return UFE_BAD_INPUT;
  }
  const int n = (int)tot;
  if ((r = dalloc(dst, &dst->d_rm_vi, n)) || (r = dalloc(dst, &dst->d_rm_w0, n)) ||
      (r = dalloc(dst, &dst->d_rm_w1x, n)) || (r = dalloc(dst, &dst->d_rm_w1y, n)))
    return r;
  HIPCHK(dst, hipMemcpyAsync(dst->d_rm_st, hst.data(), sizeof(int32_t) * nVd, hipMemcpyHostToDevice, q));
  HIPCHK(dst, hipMemcpyAsync(dst->d_rm_en, hen.data(), sizeof(int32_t) * nVd, hipMemcpyHostToDevice, q));
  k_rm_cons<<<nblk(nVd, 64), 64, 0, q>>>(R, 1, dst->d_rm_st, cnt, dst->d_rm_vi, dst->d_rm_w0, dst->d_rm_w1x,
                                         dst->d_rm_w1y, count);
  LAUNCHCHK(dst);
  // check_if_remapping_is_conservative (src/mesh_mapping_module.f90:2416-2566):
  // 2nd-order remapping of ones; interior destination vertices off by more
  // than 0.1 take triangle weights instead
  double *ones, *dx, *dy, *dd;
  HIPCHK(dst, s.alloc((void **)&ones, sizeof(double) * nVs));
  HIPCHK(dst, s.alloc((void **)&dx, sizeof(double) * nVs));
  HIPCHK(dst, s.alloc((void **)&dy, sizeof(double) * nVs));
  HIPCHK(dst, s.alloc((void **)&dd, sizeof(double) * nVd));
  k_fill<double><<<nblk(nVs), BLOCK, 0, q>>>(ones, nVs, 1.0);
  k_deriv_Aa<<<nblk(nVs), BLOCK, 0, q>>>(aa_mesh(src), ones, dx, dy);
  k_rm_apply_cons<1, true><<<layer_grid(nVd, 1, 1), BLOCK, 0, q>>>(nVd, nVs, 1, dst->d_rm_st, dst->d_rm_en, dst->d_rm_vi, dst->d_rm_w0,
                                              dst->d_rm_w1x, dst->d_rm_w1y, ones, dx, dy, dd);
  LAUNCHCHK(dst);
  std::vector<double> hd(nVd);
  HIPCHK(dst, hipMemcpyAsync(hd.data(), dd, sizeof(double) * nVd, hipMemcpyDeviceToHost, q));
  HIPCHK(dst, hipMemcpyAsync(hcount, count, sizeof(hcount), hipMemcpyDeviceToHost, q));
  HIPCHK(dst, hipStreamSynchronize(q));
  std::vector<int> wrong;
  for (int v = 0; v < nVd; v++)
    if (gd->edge_index[v] == 0 && std::fabs(1.0 - hd[v]) > 1E-1) wrong.push_back(v);
  if (!wrong.empty()) {
    std::vector<int32_t> hvi(n), htvi(3 * (size_t)nVd);
    std::vector<double> hw0(n), hw1x(n), hw1y(n);
    HIPCHK(dst, hipMemcpyAsync(hvi.data(), dst->d_rm_vi, sizeof(int32_t) * n, hipMemcpyDeviceToHost, q));
    HIPCHK(dst, hipMemcpyAsync(hw0.data(), dst->d_rm_w0, sizeof(double) * n, hipMemcpyDeviceToHost, q));
    HIPCHK(dst, hipMemcpyAsync(hw1x.data(), dst->d_rm_w1x, sizeof(double) * n, hipMemcpyDeviceToHost, q));
    HIPCHK(dst, hipMemcpyAsync(hw1y.data(), dst->d_rm_w1y, sizeof(double) * n, hipMemcpyDeviceToHost, q));
    HIPCHK(dst, hipMemcpyAsync(htvi.data(), dst->d_rm_tvi, sizeof(int32_t) * 3 * nVd, hipMemcpyDeviceToHost, q));
    HIPCHK(dst, hipStreamSynchronize(q));
    for (int v : wrong) {
      const int s0 = hst[v], ne = hen[v] - hst[v];
      if (ne < 1) continue;
      const int ia = htvi[v], ib = htvi[nVd + v], ic = htvi[2 * (size_t)nVd + v];
      const double pa[2] = {gs->V[ia - 1], gs->V[nVs + ia - 1]}, pb[2] = {gs->V[ib - 1], gs->V[nVs + ib - 1]},
                   pc[2] = {gs->V[ic - 1], gs->V[nVs + ic - 1]}, p[2] = {gd->V[v], gd->V[nVd + v]};
      const double At = rm_area_host(pa, pb, pc), Aa = rm_area_host(pb, pc, p), Ab = rm_area_host(pc, pa, p),
                   Ac = rm_area_host(pa, pb, p);
      for (int e = s0; e < hen[v]; e++) hvi[e] = 0, hw0[e] = hw1x[e] = hw1y[e] = 0.0;
      if (ne == 2) {
        if (Aa <= Ab && Aa <= Ac) {
          hvi[s0] = ib, hvi[s0 + 1] = ic, hw0[s0] = Ab / (Ab + Ac), hw0[s0 + 1] = Ac / (Ab + Ac);
        } else if (Ab <= Aa && Ab <= Ac) {
          hvi[s0] = ia, hvi[s0 + 1] = ic, hw0[s0] = Aa / (Aa + Ac), hw0[s0 + 1] = Ac / (Aa + Ac);
        } else {   // the reference lists Aa/(Aa+Ab) twice here (:2491)
          hvi[s0] = ia, hvi[s0 + 1] = ib, hw0[s0] = Aa / (Aa + Ab), hw0[s0 + 1] = Aa / (Aa + Ab);
        }
        hen[v] = s0 + 2;
      } else if (ne == 1) {
        hvi[s0] = (Aa >= Ab && Aa >= Ac) ? ia : ((Ab >= Aa && Ab >= Ac) ? ib : ic);
        hw0[s0] = 1.0;
        hen[v] = s0 + 1;
      } else {
        hvi[s0] = ia, hvi[s0 + 1] = ib, hvi[s0 + 2] = ic;
        hw0[s0] = Aa / At, hw0[s0 + 1] = Ab / At, hw0[s0 + 2] = Ac / At;
        hen[v] = s0 + 3;
      }
    }
    HIPCHK(dst, hipMemcpyAsync(dst->d_rm_vi, hvi.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, q));
    HIPCHK(dst, hipMemcpyAsync(dst->d_rm_w0, hw0.data(), sizeof(double) * n, hipMemcpyHostToDevice, q));
    HIPCHK(dst, hipMemcpyAsync(dst->d_rm_w1x, hw1x.data(), sizeof(double) * n, hipMemcpyHostToDevice, q));
    HIPCHK(dst, hipMemcpyAsync(dst->d_rm_w1y, hw1y.data(), sizeof(double) * n, hipMemcpyHostToDevice, q));
    HIPCHK(dst, hipMemcpyAsync(dst->d_rm_en, hen.data(), sizeof(int32_t) * nVd, hipMemcpyHostToDevice, q));
    HIPCHK(dst, hipStreamSynchronize(q));
  }
  ufe_remap_stats t{};
  t.n_entries = n;
  t.n_fallback = (int32_t)wrong.size();
  t.trilin_missing = hcount[RM_TRI_MISSING];
  t.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (st) *st = t;
  if ((int64_t)wrong.size() > (int64_t)std::ceil((double)nVd / 100.0)) {
    dst->err = "ufe_remap_build: 2nd order conservative remapping goes wrong for more than 1% of the vertices";
    return UFE_BAD_INPUT;
  }
  if (hcount[RM_TRI_MISSING]) {
    dst->err = "ufe_remap_build: couldnt find the source triangle containing a destination vertex";
    return UFE_BAD_INPUT;
  }
  dst->rm_nVs = nVs;
  dst->rm_nVd = nVd;
  dst->rm_n = n;
  dst->rm_ready = true;
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(dst, e.what());
} catch (...) {
  return host_failure(dst, "unknown exception");
}

int ufe_remap_field(ufe_ctx *dst, ufe_ctx *src, int method, const double *d_src, double *d_dst, int nz) {
  if (!dst || !src || !dst->rm_ready || !d_src || !d_dst || nz < 1) return UFE_BAD_INPUT;
  if (src->nV != dst->rm_nVs || dst->nV != dst->rm_nVd) {
    dst->err = "ufe_remap_field: the contexts do not hold the meshes of the remapping";
    return UFE_BAD_INPUT;
  }
  hipStream_t q = dst->stream;
  HIPCHK(dst, hipStreamSynchronize(src->stream));
  const int nVs = dst->rm_nVs, nVd = dst->rm_nVd;
  switch (method) {
    case UFE_REMAP_TRILIN:
      layered(nVd, nz, 1, [&](auto G, dim3 grid) {
        k_rm_apply_trilin<G.value><<<grid, BLOCK, 0, q>>>(nVd, nVs, nz, dst->d_rm_tvi, dst->d_rm_tw, d_src, d_dst);
      });
      break;
    case UFE_REMAP_NEAREST_NEIGHBOUR:
      layered(nVd, nz, 1, [&](auto G, dim3 grid) {
        k_rm_apply_nn<G.value><<<grid, BLOCK, 0, q>>>(nVd, nVs, nz, dst->d_rm_nn, d_src, d_dst);
      });
      break;
    case UFE_REMAP_CONS_1ST_ORDER:
      layered(nVd, nz, 1, [&](auto G, dim3 grid) {
        k_rm_apply_cons<G.value, false><<<grid, BLOCK, 0, q>>>(nVd, nVs, nz, dst->d_rm_st, dst->d_rm_en, dst->d_rm_vi,
                                                               dst->d_rm_w0, nullptr, nullptr, d_src, nullptr, nullptr,
                                                               d_dst);
      });
      break;
    case UFE_REMAP_CONS_2ND_ORDER: {
      // the derivatives' space is kept until the mesh goes (allocating and
      // freeing it took longer than the whole remapping)
      const size_t need = 2 * (size_t)nVs * nz;
      if (dst->rm_work_len < need) {
        if (dst->rm_work) HIPCHK(dst, hipFree(dst->rm_work));
        dst->rm_work = nullptr;
        dst->rm_work_len = 0;
        HIPCHK(dst, hipMalloc((void **)&dst->rm_work, sizeof(double) * need));
        dst->rm_work_len = need;
      }
      double *dx = dst->rm_work, *dy = dx + (size_t)nVs * nz;
      layered(nVs, nz, 1, [&](auto G, dim3 grid) {
        k_deriv_Aa_3D<G.value><<<grid, BLOCK, 0, q>>>(aa_mesh(src), nz, d_src, dx, dy);
      });
      layered(nVd, nz, 1, [&](auto G, dim3 grid) {
        k_rm_apply_cons<G.value, true><<<grid, BLOCK, 0, q>>>(nVd, nVs, nz, dst->d_rm_st, dst->d_rm_en, dst->d_rm_vi,
                                                              dst->d_rm_w0, dst->d_rm_w1x, dst->d_rm_w1y, d_src, dx, dy,
                                                              d_dst);
      });
      break;
    }
    default:
      dst->err = "ufe_remap_field: unknown method";
      return UFE_BAD_INPUT;
  }
  LAUNCHCHK(dst);
  HIPCHK(dst, hipStreamSynchronize(q));
  return UFE_OK;
}

int ufe_remap_ice_model(ufe_ctx *dst, ufe_ctx *src) {
  if (!dst || !src || !dst->rm_ready) return UFE_BAD_INPUT;
  if (src->nZ != dst->nZ) {
    dst->err = "ufe_remap_ice_model: the two contexts have different nZ";
    return UFE_BAD_INPUT;
  }
  int r;
  // remap_ice_model (src/ice_dynamics_module.f90:1198-1394): Hi, Hi_prev and
  // Ti conservatively (1st order); the velocities start again from zero
  if ((r = ufe_remap_field(dst, src, UFE_REMAP_CONS_1ST_ORDER, F(src, "Hi"), F(dst, "Hi"), 1))) return r;
  if ((r = ufe_remap_field(dst, src, UFE_REMAP_CONS_1ST_ORDER, F(src, "Hi_prev"), F(dst, "Hi_prev"), 1))) return r;
  if ((r = ufe_remap_field(dst, src, UFE_REMAP_CONS_1ST_ORDER, F(src, "Ti"), F(dst, "Ti"), dst->nZ))) return r;
  for (const char *f : {"U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac"})
    if ((r = ufe_field_fill(dst, field_id(f), 0.0))) return r;
  return UFE_OK;
}

int ufe_remap_export(ufe_ctx *dst, int *n_entries, int32_t *nn, int32_t *tvi, double *tw, int32_t *start,
                     int32_t *end, int32_t *vi, double *w0, double *w1x, double *w1y) {
  if (!dst || !dst->rm_ready || !n_entries) return UFE_BAD_INPUT;
  *n_entries = dst->rm_n;
  hipStream_t q = dst->stream;
  const size_t nVd = dst->rm_nVd, n = dst->rm_n;
  if (nn) HIPCHK(dst, hipMemcpyAsync(nn, dst->d_rm_nn, sizeof(int32_t) * nVd, hipMemcpyDeviceToHost, q));
  if (tvi) HIPCHK(dst, hipMemcpyAsync(tvi, dst->d_rm_tvi, sizeof(int32_t) * 3 * nVd, hipMemcpyDeviceToHost, q));
  if (tw) HIPCHK(dst, hipMemcpyAsync(tw, dst->d_rm_tw, sizeof(double) * 3 * nVd, hipMemcpyDeviceToHost, q));
  if (start) HIPCHK(dst, hipMemcpyAsync(start, dst->d_rm_st, sizeof(int32_t) * nVd, hipMemcpyDeviceToHost, q));
  if (end) HIPCHK(dst, hipMemcpyAsync(end, dst->d_rm_en, sizeof(int32_t) * nVd, hipMemcpyDeviceToHost, q));
  if (vi) HIPCHK(dst, hipMemcpyAsync(vi, dst->d_rm_vi, sizeof(int32_t) * n, hipMemcpyDeviceToHost, q));
  if (w0) HIPCHK(dst, hipMemcpyAsync(w0, dst->d_rm_w0, sizeof(double) * n, hipMemcpyDeviceToHost, q));
  if (w1x) HIPCHK(dst, hipMemcpyAsync(w1x, dst->d_rm_w1x, sizeof(double) * n, hipMemcpyDeviceToHost, q));
  if (w1y) HIPCHK(dst, hipMemcpyAsync(w1y, dst->d_rm_w1y, sizeof(double) * n, hipMemcpyDeviceToHost, q));
  HIPCHK(dst, hipStreamSynchronize(q));
  return UFE_OK;
}

// ---- mesh upload -----------------------------------------------------------
int ufe_mesh_upload(ufe_ctx *ctx, const ufe_mesh_desc *m) try {
  if (!ctx) return UFE_BAD_INPUT;
  int r = check_primary(ctx, m);
  if (r) return r;
  HIPCHK(ctx, hipSetDevice(ctx->device));
  free_mesh(ctx);
  const int nV = m->nV, nAc = m->nAc, nA = nV + nAc, nCm = m->nC_mem;
  ctx->nV = nV;
  ctx->nTri = m->nTri;
  ctx->nCm = nCm;
  ctx->nAc = nAc;
  ctx->nA = nA;
  ctx->nZ = ctx->params.nZ;
  const int64_t ldV = nV, ldA = nAc, ldAA = nA;
  // colour lists must partition the AaAc points
  {
    int64_t tot = 0;
    for (int c = 0; c < 5; c++) tot += m->colour_nV[c];
    if (tot != nA) {
      ctx->err = "colour_nV does not cover the AaAc points";
      return UFE_BAD_INPUT;
    }
  }
  // --- Aa / Ac arrays, reference layout -----------------------------------
  std::vector<int32_t> Crev((size_t)nV * nCm, 0), slot_i(nAc), slot_j(nAc);
  for (int v = 1; v <= nV; v++)
    for (int c = 1; c <= m->nC[v - 1]; c++) {
      const int vj = at(m->C, ldV, v, c);
      int found = -1;
      for (int k = 1; k <= m->nC[vj - 1]; k++)
        if (at(m->C, ldV, vj, k) == v) { found = k - 1; break; }
      if (found < 0) {
        ctx->err = "connectivity is not symmetric";
        return UFE_BAD_INPUT;
      }
      Crev[(size_t)(c - 1) * nV + (v - 1)] = found;
    }
  for (int a = 1; a <= nAc; a++) {
    const int vi = at(m->Aci, ldA, a, 1), vj = at(m->Aci, ldA, a, 2);
    int ci = -1, cj = -1;
    for (int k = 1; k <= m->nC[vi - 1]; k++) if (at(m->C, ldV, vi, k) == vj) { ci = k - 1; break; }
    for (int k = 1; k <= m->nC[vj - 1]; k++) if (at(m->C, ldV, vj, k) == vi) { cj = k - 1; break; }
    if (ci < 0 || cj < 0) {
      ctx->err = "Aci does not match the connectivity";
      return UFE_BAD_INPUT;
    }
    slot_i[a - 1] = ci;
    slot_j[a - 1] = cj;
  }
  const size_t w1 = (size_t)nV * (nCm + 1);
  if ((r = dupload(ctx, &ctx->d_nC, m->nC, nV))) return r;
  if ((r = dupload(ctx, &ctx->d_C, m->C, (size_t)nV * nCm))) return r;
  if ((r = dupload(ctx, &ctx->d_edge, m->edge_index, nV))) return r;
  if ((r = dupload(ctx, &ctx->d_iAci, (const int32_t *)m->iAci, (size_t)nV * nCm))) return r;
  if ((r = dupload(ctx, &ctx->d_Crev, Crev.data(), Crev.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_Nx, (const double *)m->Nx, w1))) return r;
  if ((r = dupload(ctx, &ctx->d_Ny, (const double *)m->Ny, w1))) return r;
  if ((r = dupload(ctx, &ctx->d_Nxx, (const double *)m->Nxx, w1))) return r;
  if ((r = dupload(ctx, &ctx->d_Nxy, (const double *)m->Nxy, w1))) return r;
  if ((r = dupload(ctx, &ctx->d_Nyy, (const double *)m->Nyy, w1))) return r;
  if (m->A) {
    if ((r = dupload(ctx, &ctx->d_A, m->A, nV))) return r;
  } else if ((r = dalloc(ctx, &ctx->d_A, nV))) return r;
  if (m->Cw) {
    if ((r = dupload(ctx, &ctx->d_Cw, m->Cw, (size_t)nV * nCm))) return r;
  } else if ((r = dalloc(ctx, &ctx->d_Cw, (size_t)nV * nCm))) return r;
  if ((r = dupload(ctx, &ctx->d_V, m->V, (size_t)nV * 2))) return r;
  if ((r = dupload(ctx, &ctx->d_Aci, (const int32_t *)m->Aci, (size_t)nAc * 4))) return r;
  if ((r = dupload(ctx, &ctx->d_edgeAc, (const int32_t *)m->edge_index_Ac, nAc))) return r;
  if ((r = dupload(ctx, &ctx->d_slot_i, slot_i.data(), nAc))) return r;
  if ((r = dupload(ctx, &ctx->d_slot_j, slot_j.data(), nAc))) return r;
  if ((r = dupload(ctx, &ctx->d_NxAc, (const double *)m->Nx_Ac, (size_t)nAc * 4))) return r;
  if ((r = dupload(ctx, &ctx->d_NyAc, (const double *)m->Ny_Ac, (size_t)nAc * 4))) return r;
  if ((r = dupload(ctx, &ctx->d_NoAc, (const double *)m->No_Ac, (size_t)nAc * 4))) return r;
  if ((r = dupload(ctx, &ctx->d_NpAc, (const double *)m->Np_Ac, nAc))) return r;

  // --- colour order -------------------------------------------------------
  auto is_edge = [&](int ai1) {
    return ai1 <= nV ? m->edge_index[ai1 - 1] > 0 : m->edge_index_Ac[ai1 - nV - 1] > 0;
  };
  // Inside a colour the update order is free (same-colour points are never
  // neighbours), so rows are sorted along a Hilbert curve of their
  // coordinates: a wavefront then works on a compact patch and its
  // neighbour gathers from the other colours hit few cache lines.
  std::vector<uint64_t> hkey(nA);
  {
    const double span = std::max(m->xmax - m->xmin, m->ymax - m->ymin);
    for (int a = 0; a < nA; a++) {
      const double fx = (at(m->VAaAc, ldAA, a + 1, 1) - m->xmin) / span;
      const double fy = (at(m->VAaAc, ldAA, a + 1, 2) - m->ymin) / span;
      const uint32_t gx = (uint32_t)std::min(65535.0, std::max(0.0, fx * 65535.0));
      const uint32_t gy = (uint32_t)std::min(65535.0, std::max(0.0, fy * 65535.0));
      hkey[a] = hilbert_index(gx, gy);
    }
  }
  // member of each AaAc point when a batch was declared for this mesh
  std::vector<int32_t> member;
  if (!ctx->b_nV.empty()) {
    int64_t sv = 0, sa = 0;
    for (size_t b = 0; b < ctx->b_nV.size(); b++) {
      sv += ctx->b_nV[b];
      sa += ctx->b_nAc[b];
    }
    if (sv != nV || sa != nAc) {
      ctx->err = "the declared batch does not add up to the uploaded mesh";
      return UFE_BAD_INPUT;
    }
    member.resize(nA);
    int a = 0;
    for (size_t b = 0; b < ctx->b_nV.size(); b++)
      for (int k = 0; k < ctx->b_nV[b]; k++) member[a++] = (int32_t)b;
    for (size_t b = 0; b < ctx->b_nAc.size(); b++)
      for (int k = 0; k < ctx->b_nAc[b]; k++) member[a++] = (int32_t)b;
  }
  std::vector<int32_t> perm;
  perm.reserve(nA);
  for (int c = 1; c <= 5; c++) {
    ctx->colour_start[c - 1] = (int)perm.size();
    std::vector<int32_t> act, edg;
    for (int k = 1; k <= m->colour_nV[c - 1]; k++) {
      const int ai = at(m->colour_vi, ldAA, k, c);
      if (ai < 1 || ai > nA) {
        ctx->err = "colour_vi holds an index outside 1..nVAaAc";
        return UFE_BAD_INPUT;
      }
      (is_edge(ai) ? edg : act).push_back(ai - 1);
    }
    auto by_key = [&](int32_t a, int32_t b) {
      if (!member.empty() && member[a] != member[b]) return member[a] < member[b];
      return hkey[a] < hkey[b] || (hkey[a] == hkey[b] && a < b);
    };
    std::sort(act.begin(), act.end(), by_key);
    perm.insert(perm.end(), act.begin(), act.end());
    perm.insert(perm.end(), edg.begin(), edg.end());
    ctx->colour_active[c - 1] = (int)act.size();
  }
  ctx->colour_start[5] = nA;
  if ((int)perm.size() != nA) {
    ctx->err = "colour lists are not a partition";
    return UFE_BAD_INPUT;
  }
  std::vector<int32_t> iperm(nA, -1);
  for (int p = 0; p < nA; p++) {
    if (iperm[perm[p]] != -1) {
      ctx->err = "colour lists repeat a point";
      return UFE_BAD_INPUT;
    }
    iperm[perm[p]] = p;
  }
  // SELL-64 arrays over the colour order
  const int nchunk = (nA + SELL - 1) / SELL;
  std::vector<int64_t> cptr(nchunk + 1, 0);
  std::vector<int32_t> cw(nchunk, 0);
  std::vector<uint8_t> deg(nA);
  for (int p = 0; p < nA; p++) {
    const int n = m->nCAaAc[perm[p]];
    if (n < 2 || n > nCm) {
      ctx->err = "nCAaAc out of range";
      return UFE_BAD_INPUT;
    }
    deg[p] = (uint8_t)n;
    cw[p / SELL] = std::max(cw[p / SELL], n);
  }
  for (int k = 0; k < nchunk; k++) cptr[k + 1] = cptr[k] + (int64_t)cw[k] * SELL;
  const int64_t ne = cptr[nchunk];
  std::vector<int32_t> col(ne);
  std::vector<double> cNx(ne, 0.0), cNy(ne, 0.0);
  std::vector<double2> cU(ne, make_double2(0.0, 0.0));
  std::vector<double> hNx(nA), hNy(nA), hNxx(nA), hNyy(nA), Sxx(nA), Sxy(nA), Syy(nA);
  for (int p = 0; p < nA; p++) {
    const int ai = perm[p] + 1, n = deg[p];
    const int64_t base = cptr[p / SELL] + (p % SELL);
    for (int s = 0; s < cw[p / SELL]; s++) col[base + (int64_t)s * SELL] = p;
    for (int s = 1; s <= n; s++) {
      const int64_t e = base + (int64_t)(s - 1) * SELL;
      col[e] = iperm[at(m->CAaAc, ldAA, ai, s) - 1];
      cNx[e] = at(m->Nx_AaAc, ldAA, ai, s);
      cNy[e] = at(m->Ny_AaAc, ldAA, ai, s);
      const double nxx = at(m->Nxx_AaAc, ldAA, ai, s), nyy = at(m->Nyy_AaAc, ldAA, ai, s);
      cU[e] = make_double2(4.0 * nxx + nyy, 4.0 * nyy + nxx);
    }
    hNx[p] = at(m->Nx_AaAc, ldAA, ai, n + 1);
    hNy[p] = at(m->Ny_AaAc, ldAA, ai, n + 1);
    hNxx[p] = at(m->Nxx_AaAc, ldAA, ai, n + 1);
    hNyy[p] = at(m->Nyy_AaAc, ldAA, ai, n + 1);
    double a = at(m->Nxx_AaAc, ldAA, ai, n + 1), b = at(m->Nxy_AaAc, ldAA, ai, n + 1),
           c = at(m->Nyy_AaAc, ldAA, ai, n + 1);
    for (int s = 1; s <= n; s++) {
      a = a + at(m->Nxx_AaAc, ldAA, ai, s);
      b = b + at(m->Nxy_AaAc, ldAA, ai, s);
      c = c + at(m->Nyy_AaAc, ldAA, ai, s);
    }
    Sxx[p] = a;
    Sxy[p] = b;
    Syy[p] = c;
  }
  // Neumann lists: edge points average their non-edge neighbours; the domain
  // corners (vertices 1..4 of a reference mesh, the only points with the
  // corner codes 2/4/6/8 in edge_index) then average all their neighbours.
  auto is_corner = [&](int ai) {
    if (ai > nV) return false;
    const int e = m->edge_index[ai - 1];
    return e == 2 || e == 4 || e == 6 || e == 8;
  };
  if (member.empty())
    for (int ai = 1; ai <= nV; ai++)
      if (is_corner(ai) != (ai <= 4)) {
        ctx->err = "vertices 1..4 must be the domain corners (edge_index 2/4/6/8), and only they";
        return UFE_BAD_INPUT;
      }
  std::vector<int32_t> nrow, nptr{0}, ncol, crow, cptr2{0}, ccol;
  for (int ai = 1; ai <= nA; ai++) {
    if (!is_edge(ai) || is_corner(ai)) continue;
    nrow.push_back(iperm[ai - 1]);
    int cnt = 0;
    for (int s = 1; s <= m->nCAaAc[ai - 1]; s++) {
      const int aj = at(m->CAaAc, ldAA, ai, s);
      if (is_edge(aj)) continue;
      ncol.push_back(iperm[aj - 1]);
      cnt++;
    }
    if (cnt == 0) {
      ctx->err = "an edge point has no non-edge neighbour (Neumann mean undefined)";
      return UFE_BAD_INPUT;
    }
    nptr.push_back((int32_t)ncol.size());
  }
  for (int ai = 1; ai <= nV; ai++) {
    if (!is_corner(ai)) continue;
    crow.push_back(iperm[ai - 1]);
    for (int s = 1; s <= m->nCAaAc[ai - 1]; s++) ccol.push_back(iperm[at(m->CAaAc, ldAA, ai, s) - 1]);
    cptr2.push_back((int32_t)ccol.size());
  }
  // transposed slot coefficients: row q, slot s, neighbour p = col[q,s]: the
  // coefficient of q in p's equation (zero when p is an edge row)
  std::vector<uint8_t> active(nA, 0);
  for (int c = 0; c < 5; c++)
    for (int p = ctx->colour_start[c]; p < ctx->colour_start[c] + ctx->colour_active[c]; p++) active[p] = 1;
  std::vector<double2> cUT(ne, make_double2(0.0, 0.0));
  std::vector<double> cNxT(ne, 0.0), cNyT(ne, 0.0);
  for (int q = 0; q < nA; q++) {
    const int64_t bq = cptr[q / SELL] + (q % SELL);
    for (int s = 0; s < deg[q]; s++) {
      const int64_t e = bq + (int64_t)s * SELL;
      const int p = col[e];
      if (!active[p]) continue;
      const int64_t bp = cptr[p / SELL] + (p % SELL);
      int64_t f = -1;
      for (int t = 0; t < deg[p]; t++)
        if (col[bp + (int64_t)t * SELL] == q) { f = bp + (int64_t)t * SELL; break; }
      if (f < 0) {
        ctx->err = "AaAc connectivity is not symmetric";
        return UFE_BAD_INPUT;
      }
      cUT[e] = cU[f];
      cNxT[e] = cNx[f];
      cNyT[e] = cNy[f];
    }
  }
  // reverse edge-average lists: SOR row a <- edge rows whose mean includes a
  std::vector<std::vector<std::pair<int32_t, int32_t>>> rev(nA);
  for (size_t i = 0; i < nrow.size(); i++)
    for (int k = nptr[i]; k < nptr[i + 1]; k++)
      rev[ncol[k]].push_back({nrow[i], nptr[i + 1] - nptr[i]});
  std::vector<int32_t> rtgt, rptr{0}, rsrc, rcnt;
  for (int a = 0; a < nA; a++) {
    if (rev[a].empty()) continue;
    if (!active[a]) {
      ctx->err = "an edge point averages another edge point";
      return UFE_BAD_INPUT;
    }
    rtgt.push_back(a);
    for (auto &pr : rev[a]) {
      rsrc.push_back(pr.first);
      rcnt.push_back(pr.second);
    }
    rptr.push_back((int32_t)rsrc.size());
  }
  ctx->n_rev = (int)rtgt.size();
  if ((r = dupload(ctx, &ctx->d_cUT, cUT.data(), cUT.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cNxT, cNxT.data(), cNxT.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cNyT, cNyT.data(), cNyT.size()))) return r;
  if (ctx->n_rev) {
    if ((r = dupload(ctx, &ctx->d_rev_tgt, rtgt.data(), rtgt.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_rev_ptr, rptr.data(), rptr.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_rev_src, rsrc.data(), rsrc.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_rev_cnt, rcnt.data(), rcnt.size()))) return r;
  }
  ctx->n_neu = (int)nrow.size();
  ctx->n_cor = (int)crow.size();
  ctx->h_perm = perm;
  ctx->h_key.resize(nA);
  for (int p = 0; p < nA; p++) ctx->h_key[p] = (uint32_t)hkey[perm[p]];
  if ((r = dupload(ctx, &ctx->d_perm, perm.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_iperm, iperm.data(), nA))) return r;
  {
    std::vector<uint8_t> none(nA, 0);
    if ((r = dupload(ctx, &ctx->d_skip, none.data(), nA))) return r;
  }
  if ((r = dupload(ctx, &ctx->d_chunk_ptr, cptr.data(), cptr.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_chunk_w, cw.data(), cw.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_deg, deg.data(), deg.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_col, col.data(), col.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cNx, cNx.data(), cNx.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cNy, cNy.data(), cNy.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cU, cU.data(), cU.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_hNx, hNx.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_hNy, hNy.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_hNxx, hNxx.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_hNyy, hNyy.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_Sxx, Sxx.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_Sxy, Sxy.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_Syy, Syy.data(), nA))) return r;
  if ((r = dupload(ctx, &ctx->d_neu_row, nrow.data(), nrow.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_neu_ptr, nptr.data(), nptr.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_neu_col, ncol.data(), ncol.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cor_row, crow.data(), crow.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cor_ptr, cptr2.data(), cptr2.size()))) return r;
  if ((r = dupload(ctx, &ctx->d_cor_col, ccol.data(), ccol.size()))) return r;

  // --- FP32 copies and algorithmic bytes ---------------------------------
  {
    std::vector<float2> cU32(ne);
    for (int64_t e = 0; e < ne; e++) cU32[e] = make_float2((float)cU[e].x, (float)cU[e].y);
    std::vector<float> Sxy32(nA);
    for (int p = 0; p < nA; p++) Sxy32[p] = (float)Sxy[p];
    if ((r = dupload(ctx, &ctx->d_cU32, cU32.data(), cU32.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_Sxy32, Sxy32.data(), Sxy32.size()))) return r;
    if ((r = dalloc(ctx, &ctx->d_EV32, nA))) return r;
    if ((r = dalloc(ctx, &ctx->d_R32, nA))) return r;
    HIPCHK(ctx, hipMemsetAsync(ctx->d_R32, 0, sizeof(float2) * nA, ctx->stream));
    if ((r = dalloc(ctx, &ctx->d_D32, nA))) return r;
    ctx->degsum = 0.0;
    for (int c = 0; c < 5; c++) {
      double b64 = 0.0, b32 = 0.0;
      for (int p = ctx->colour_start[c]; p < ctx->colour_start[c] + ctx->colour_active[c]; p++) {
        const double n = deg[p];
        b64 += 4.0 * (n + 1.0) + 8.0 * (2.0 * n + 9.0);
        b32 += 4.0 * (n + 1.0) + 4.0 * (2.0 * n + 9.0);
        ctx->degsum += n;
      }
      ctx->bytes64[c] = b64;
      ctx->bytes32[c] = b32;
    }
  }

  // --- fields (zero-initialised, like the reference's shared windows) ------
  ctx->field_ptr.assign(NFIELDS, nullptr);
  for (int i = 0; i < NFIELDS; i++) {
    if (FIELDS[i].pair >= 0) continue;
    const size_t n = grid_len(ctx, FIELDS[i].grid);
    if (FIELDS[i].dtype == D_F64) {
      double *p;
      if ((r = dalloc(ctx, &p, n))) return r;
      HIPCHK(ctx, hipMemsetAsync(p, 0, n * sizeof(double), ctx->stream));
      ctx->field_ptr[i] = p;
    } else {
      int32_t *p;
      if ((r = dalloc(ctx, &p, n))) return r;
      HIPCHK(ctx, hipMemsetAsync(p, 0, n * sizeof(int32_t), ctx->stream));
      ctx->field_ptr[i] = p;
    }
  }
  for (int k = 0; k < 3; k++) {
    if ((r = dalloc(ctx, &ctx->d_pair[k], nA))) return r;
    HIPCHK(ctx, hipMemsetAsync(ctx->d_pair[k], 0, sizeof(double2) * nA, ctx->stream));
  }
  ctx->n_part = nblk(std::max(nA, nV)) + 16;
  if ((r = dalloc(ctx, &ctx->d_part, 2 * (size_t)ctx->n_part))) return r;
  if ((r = dalloc(ctx, &ctx->d_scalar, 8))) return r;
  for (int k = 0; k < 4; k++)
    if ((r = dalloc(ctx, &ctx->d_tmp[k], (size_t)std::max(nA, nV * std::max(ctx->nZ, nCm))))) return r;
  if ((r = dalloc(ctx, &ctx->d_ViSMB, nV))) return r;
  if ((r = dalloc(ctx, &ctx->d_count, 4))) return r;
  if ((r = dalloc(ctx, &ctx->d_flags, 1))) return r;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  // --- batch tables: member of each row and SOR-row chunks inside one member
  if (!member.empty()) {
    const int nbm = (int)ctx->b_nV.size();
    std::vector<uint16_t> mid(nA);
    for (int p = 0; p < nA; p++) mid[p] = (uint16_t)member[perm[p]];
    constexpr int CH = 4096;
    std::vector<std::vector<std::pair<int32_t, int32_t>>> per(nbm);
    ctx->b_rows.assign(nbm, 0);
    for (int c = 0; c < 5; c++) {
      const int s0 = ctx->colour_start[c], e0 = s0 + ctx->colour_active[c];
      for (int p = s0; p < e0;) {
        const int b = mid[p];
        int q = p;
        while (q < e0 && mid[q] == b && q - p < CH) q++;
        per[b].push_back({p, q - p});
        ctx->b_rows[b] += q - p;
        p = q;
      }
    }
    std::vector<int32_t> cs, cc, cm, mptr{0};
    for (int b = 0; b < nbm; b++) {
      if (per[b].empty()) {
        ctx->err = "a batch member has no SOR rows";
        return UFE_BAD_INPUT;
      }
      for (auto &x : per[b]) {
        cs.push_back(x.first);
        cc.push_back(x.second);
        cm.push_back(b);
      }
      mptr.push_back((int32_t)cs.size());
    }
    ctx->n_chunk = (int)cs.size();
    ctx->h_mch_ptr = mptr;
    ctx->h_mid = mid;
    if ((r = dupload(ctx, &ctx->d_mid, mid.data(), mid.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_ch_start, cs.data(), cs.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_ch_count, cc.data(), cc.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_ch_member, cm.data(), cm.size()))) return r;
    if ((r = dupload(ctx, &ctx->d_mch_ptr, mptr.data(), mptr.size()))) return r;
    ctx->nb = nbm;
  }
  // triangles for the upwind derivatives, their neighbour functions
  // (src/mesh_derivatives_module.f90:30-47) and the resolution R
  // (src/mesh_help_functions_module.f90:193-216)
  if ((r = dupload(ctx, &ctx->d_Tri, m->Tri, (size_t)m->nTri * 3))) return r;
  if ((r = dupload(ctx, &ctx->d_niTri, m->niTri, nV))) return r;
  if ((r = dupload(ctx, &ctx->d_iTri, m->iTri, (size_t)nV * nCm))) return r;
  if ((r = dalloc(ctx, &ctx->d_NxTri, (size_t)m->nTri * 3))) return r;
  if ((r = dalloc(ctx, &ctx->d_NyTri, (size_t)m->nTri * 3))) return r;
  if ((r = dalloc(ctx, &ctx->d_R, nV))) return r;
  if ((r = dalloc(ctx, &ctx->d_crit, 3 * (size_t)CRIT_MAX_BLOCKS + 3))) return r;
  if ((r = dalloc(ctx, &ctx->d_icount, 4))) return r;
  {
    TriMesh t = tri_mesh(ctx);
    k_tri_neighbour_functions<<<nblk(m->nTri), BLOCK, 0, ctx->stream>>>(t);
    GeomMesh g{};
    g.nV = nV;
    g.xmin = m->xmin;
    g.xmax = m->xmax;
    g.V = ctx->d_V;
    g.nC = ctx->d_nC;
    g.C = ctx->d_C;
    k_geo_resolution<<<nblk(nV), BLOCK, 0, ctx->stream>>>(g, ctx->d_R);
    LAUNCHCHK(ctx);
  }
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  ctx->have_mesh = true;
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

// ---- fields ----------------------------------------------------------------
static int field_xfer(ufe_ctx *ctx, int id, void *buf, bool to_dev, bool buf_is_dev) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  if (id < 0 || id >= NFIELDS || !buf) {
    ctx->err = "bad field id or buffer";
    return UFE_BAD_INPUT;
  }
  const FieldDef &fd = FIELDS[id];
  const size_t n = grid_len(ctx, fd.grid);
  const size_t bytes = n * (fd.dtype == D_F64 ? 8 : 4);
  const hipMemcpyKind k_in = buf_is_dev ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
  const hipMemcpyKind k_out = buf_is_dev ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
  if (fd.grid != G_AAAC) {
    void *d = ctx->field_ptr[id];
    if (to_dev) HIPCHK(ctx, hipMemcpyAsync(d, buf, bytes, k_in, ctx->stream));
    else HIPCHK(ctx, hipMemcpyAsync(buf, d, bytes, k_out, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return UFE_OK;
  }
  double *tmp = ctx->d_tmp[3];
  if (to_dev) {
    HIPCHK(ctx, hipMemcpyAsync(tmp, buf, bytes, k_in, ctx->stream));
    if (fd.pair >= 0)
      k_gather_perm_pair<<<nblk(n), BLOCK, 0, ctx->stream>>>((int)n, ctx->d_perm, tmp, ctx->d_pair[fd.pair], fd.comp);
    else
      k_gather_perm<<<nblk(n), BLOCK, 0, ctx->stream>>>((int)n, ctx->d_perm, tmp, (double *)ctx->field_ptr[id]);
    LAUNCHCHK(ctx);
  } else {
    if (fd.pair >= 0)
      k_scatter_perm_pair<<<nblk(n), BLOCK, 0, ctx->stream>>>((int)n, ctx->d_perm, ctx->d_pair[fd.pair], tmp, fd.comp);
    else
      k_scatter_perm<<<nblk(n), BLOCK, 0, ctx->stream>>>((int)n, ctx->d_perm, (const double *)ctx->field_ptr[id], tmp);
    LAUNCHCHK(ctx);
    HIPCHK(ctx, hipMemcpyAsync(buf, tmp, bytes, k_out, ctx->stream));
  }
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

int ufe_field_set(ufe_ctx *ctx, int id, const void *host) { return field_xfer(ctx, id, (void *)host, true, false); }
int ufe_field_get(ufe_ctx *ctx, int id, void *host) { return field_xfer(ctx, id, host, false, false); }
int ufe_field_set_device(ufe_ctx *ctx, int id, const void *dev) { return field_xfer(ctx, id, (void *)dev, true, true); }
int ufe_field_get_device(ufe_ctx *ctx, int id, void *dev) { return field_xfer(ctx, id, dev, false, true); }

// ---- update_general_ice_model_data ------------------------------------------
static GenFields gen_fields(ufe_ctx *c) {
  GenFields f;
  f.Hi = F(c, "Hi"); f.Hb = F(c, "Hb"); f.SL = F(c, "SL"); f.dHb_dt = F(c, "dHb_dt"); f.dHi_dt = F(c, "dHi_dt");
  f.Hs = F(c, "Hs"); f.dHs_dt = F(c, "dHs_dt"); f.dHi_dx = F(c, "dHi_dx"); f.dHi_dy = F(c, "dHi_dy");
  f.dHs_dx = F(c, "dHs_dx"); f.dHs_dy = F(c, "dHs_dy"); f.dHs_dx_shelf = F(c, "dHs_dx_shelf");
  f.dHs_dy_shelf = F(c, "dHs_dy_shelf");
  f.land = FI(c, "mask_land"); f.ocean = FI(c, "mask_ocean"); f.lake = FI(c, "mask_lake");
  f.ice = FI(c, "mask_ice"); f.sheet = FI(c, "mask_sheet"); f.shelf = FI(c, "mask_shelf");
  f.coast = FI(c, "mask_coast"); f.margin = FI(c, "mask_margin"); f.gl = FI(c, "mask_gl");
  f.cf = FI(c, "mask_cf"); f.mask = FI(c, "mask");
  f.Hi_Ac = F(c, "Hi_Ac"); f.Hb_Ac = F(c, "Hb_Ac"); f.SL_Ac = F(c, "SL_Ac"); f.Hs_Ac = F(c, "Hs_Ac");
  f.dHi_dx_Ac = F(c, "dHi_dx_Ac"); f.dHi_dy_Ac = F(c, "dHi_dy_Ac"); f.dHi_dp_Ac = F(c, "dHi_dp_Ac");
  f.dHi_do_Ac = F(c, "dHi_do_Ac"); f.dHb_dx_Ac = F(c, "dHb_dx_Ac"); f.dHb_dy_Ac = F(c, "dHb_dy_Ac");
  f.dHb_dp_Ac = F(c, "dHb_dp_Ac"); f.dHb_do_Ac = F(c, "dHb_do_Ac"); f.dHs_dx_Ac = F(c, "dHs_dx_Ac");
  f.dHs_dy_Ac = F(c, "dHs_dy_Ac"); f.dHs_dp_Ac = F(c, "dHs_dp_Ac"); f.dHs_do_Ac = F(c, "dHs_do_Ac");
  f.dSL_dx_Ac = F(c, "dSL_dx_Ac"); f.dSL_dy_Ac = F(c, "dSL_dy_Ac"); f.dSL_dp_Ac = F(c, "dSL_dp_Ac");
  f.dSL_do_Ac = F(c, "dSL_do_Ac"); f.dHs_dx_shelf_Ac = F(c, "dHs_dx_shelf_Ac");
  f.dHs_dy_shelf_Ac = F(c, "dHs_dy_shelf_Ac");
  f.landA = FI(c, "mask_land_Ac"); f.oceanA = FI(c, "mask_ocean_Ac"); f.lakeA = FI(c, "mask_lake_Ac");
  f.iceA = FI(c, "mask_ice_Ac"); f.sheetA = FI(c, "mask_sheet_Ac"); f.shelfA = FI(c, "mask_shelf_Ac");
  f.coastA = FI(c, "mask_coast_Ac"); f.marginA = FI(c, "mask_margin_Ac"); f.glA = FI(c, "mask_gl_Ac");
  f.cfA = FI(c, "mask_cf_Ac"); f.maskA = FI(c, "mask_Ac");
  return f;
}

static int enqueue_physical_properties(ufe_ctx *ctx, int mode) {
  PhysParams p;
  p.nZ = ctx->nZ;
  p.mode = mode;
  for (int k = 0; k < ctx->nZ; k++) p.zeta[k] = ctx->params.zeta[k];
  k_phys_aa<<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(ctx->nV, p, F(ctx, "Ti"), F(ctx, "Hi"),
                                                       FI(ctx, "mask_sheet"), F(ctx, "A_flow"),
                                                       F(ctx, "A_flow_mean"), F(ctx, "Ti_pmp"),
                                                       F(ctx, "Cpi"), F(ctx, "Ki"));
  k_phys_ac<<<nblk(ctx->nAc), BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), p, F(ctx, "Ti"), FI(ctx, "mask_sheet_Ac"),
                                                        F(ctx, "Ti_Ac"), F(ctx, "A_flow_Ac"),
                                                        F(ctx, "A_flow_mean_Ac"));
  LAUNCHCHK(ctx);
  return UFE_OK;
}

static bool phys_mode_ok(int mode) {
  return mode == UFE_PHYS_ARRHENIUS || mode == UFE_PHYS_BENCHMARK_FIXED;
}

int ufe_update_general_ice_model_data(ufe_ctx *ctx) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  const int mode = ctx->params.physical_properties;
  if (mode != UFE_PHYS_INPUT && !phys_mode_ok(mode)) {
    ctx->err = "physical_properties must be UFE_PHYS_INPUT, UFE_PHYS_ARRHENIUS or UFE_PHYS_BENCHMARK_FIXED";
    return UFE_BAD_INPUT;
  }
  GenFields f = gen_fields(ctx);
  k_gen_ac<<<xcd_grid(ctx->nAc), BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), f);
  k_gen_aa<<<xcd_grid(ctx->nV), BLOCK, 0, ctx->stream>>>(aa_mesh(ctx), f);
  LAUNCHCHK(ctx);
  // ice_physical_properties closes the routine (src/general_ice_model_data_module.f90:91)
  if (mode != UFE_PHYS_INPUT) {
    const int st = enqueue_physical_properties(ctx, mode);
    if (st != UFE_OK) return st;
  }
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

int ufe_ice_physical_properties(ufe_ctx *ctx, int mode) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  if (!phys_mode_ok(mode)) {
    ctx->err = "ufe_ice_physical_properties: mode must be UFE_PHYS_ARRHENIUS or UFE_PHYS_BENCHMARK_FIXED";
    return UFE_BAD_INPUT;
  }
  const int st = enqueue_physical_properties(ctx, mode);
  if (st != UFE_OK) return st;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

// ---- solve_SIA ---------------------------------------------------------------
int ufe_solve_SIA(ufe_ctx *ctx) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  SIAParams p;
  p.nZ = ctx->nZ;
  p.m_enh = ctx->params.m_enh_sia;
  for (int k = 0; k < ctx->nZ; k++) {
    p.zeta[k] = ctx->params.zeta[k];
    p.zeta_n[k] = std::pow(ctx->params.zeta[k], N_FLOW);
  }
  auto sia = [&](auto kernel) {
    kernel<<<nblk(ctx->nAc), BLOCK, 0, ctx->stream>>>(
        ctx->nAc, p, F(ctx, "Hi_Ac"), F(ctx, "dHs_dx_Ac"), F(ctx, "dHs_dy_Ac"), F(ctx, "dHs_dp_Ac"),
        F(ctx, "dHs_do_Ac"), FI(ctx, "mask_sheet_Ac"), F(ctx, "A_flow_Ac"), F(ctx, "D_SIA_3D_Ac"),
        F(ctx, "D_SIA_Ac"), F(ctx, "Ux_SIA_Ac"), F(ctx, "Uy_SIA_Ac"), F(ctx, "Up_SIA_Ac"), F(ctx, "Uo_SIA_Ac"));
  };
  if (p.nZ <= COLUMN_REGS) sia(k_sia<COLUMN_REGS>);
  else sia(k_sia<MAX_NZ>);
  k_map3_Ac_to_Aa<<<xcd_grid(ctx->nV), BLOCK, 0, ctx->stream>>>(aa_mesh(ctx), F(ctx, "Ux_SIA_Ac"), F(ctx, "Uy_SIA_Ac"),
                                                               F(ctx, "D_SIA_Ac"), F(ctx, "U_SIA"), F(ctx, "V_SIA"),
                                                               F(ctx, "D_SIA"));
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

// ---- solve_SIA_3D and the critical time steps ---------------------------------
// apply_Neumann_boundary_3D of one or two fields
static void neumann_Aa(ufe_ctx *ctx, int nz, double *d0, double *d1 = nullptr) {
  const int fields = d1 ? 2 : 1;
  layered(ctx->nV, nz, fields, [&](auto G, dim3 grid) {
    k_neumann_Aa_edges<G.value><<<grid, BLOCK, 0, ctx->stream>>>(aa_mesh(ctx), nz, d0, d1);
  });
  k_neumann_Aa_corners<<<dim3(nblk(nz, 64), fields), 64, 0, ctx->stream>>>(aa_mesh(ctx), nz, d0, d1);
}

int ufe_solve_SIA_3D(ufe_ctx *ctx) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  SIA3DParams p;
  p.nZ = ctx->nZ;
  p.m_enh = ctx->params.m_enh_sia;
  for (int k = 0; k < ctx->nZ; k++) {
    p.zeta[k] = ctx->params.zeta[k];
    p.zeta_n[k] = std::pow(ctx->params.zeta[k], N_FLOW);
  }
  SIA3DFields f;
  f.Hi = F(ctx, "Hi");
  f.Af = F(ctx, "A_flow");
  f.Us = F(ctx, "U_SSA");
  f.Vs = F(ctx, "V_SSA");
  f.sx = F(ctx, "dHs_dx");
  f.sy = F(ctx, "dHs_dy");
  f.ix = F(ctx, "dHi_dx");
  f.iy = F(ctx, "dHi_dy");
  f.dHb_dt = F(ctx, "dHb_dt");
  f.shelf = FI(ctx, "mask_shelf");
  f.sheet = FI(ctx, "mask_sheet");
  f.U3 = F(ctx, "U_3D");
  f.V3 = F(ctx, "V_3D");
  f.W3 = F(ctx, "W_3D");
  const AaMesh am = aa_mesh(ctx);
  const int nz = ctx->nZ;
  hipStream_t q = ctx->stream;
  if (nz <= COLUMN_REGS) k_sia3d_uv<COLUMN_REGS><<<nblk(ctx->nV), BLOCK, 0, q>>>(ctx->nV, p, f);
  else k_sia3d_uv<MAX_NZ><<<nblk(ctx->nV), BLOCK, 0, q>>>(ctx->nV, p, f);
  neumann_Aa(ctx, nz, f.U3, f.V3);   // apply_Neumann_boundary_3D (:366-367)
  k_sia3d_w<<<xcd_grid(ctx->nV), BLOCK, 0, q>>>(am, p, f);
  neumann_Aa(ctx, nz, f.W3);
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipStreamSynchronize(q));
  return UFE_OK;
}

int ufe_critical_timesteps(ufe_ctx *ctx, double *dt_crit) {
  if (!ctx || !ctx->have_mesh || !dt_crit) return UFE_BAD_INPUT;
  const int n = std::max(ctx->nAc, ctx->nV);
  const int nb = std::max(1, std::min(CRIT_MAX_BLOCKS, (n + CRIT_BLOCK - 1) / CRIT_BLOCK));
  hipStream_t q = ctx->stream;
  double *out = ctx->d_crit + 3 * (size_t)CRIT_MAX_BLOCKS;
  k_crit_partial<<<nb, CRIT_BLOCK, 0, q>>>(ac_mesh(ctx), ctx->d_A, ctx->nZ, F(ctx, "D_SIA_Ac"), F(ctx, "U_SSA"),
                                           F(ctx, "V_SSA"), F(ctx, "U_3D"), F(ctx, "V_3D"), ctx->d_crit);
  k_crit_finish<<<1, CRIT_BLOCK, 0, q>>>(nb, ctx->d_crit, out);
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipMemcpyAsync(dt_crit, out, 3 * sizeof(double), hipMemcpyDeviceToHost, q));
  HIPCHK(ctx, hipStreamSynchronize(q));
  return UFE_OK;
}

// ---- SOR ---------------------------------------------------------------------
static NeumannList neu_list(ufe_ctx *c) {
  NeumannList L;
  L.n = c->n_neu;
  L.row = c->d_neu_row;
  L.ptr = c->d_neu_ptr;
  L.col = c->d_neu_col;
  return L;
}
static NeumannList cor_list(ufe_ctx *c) {
  NeumannList L;
  L.n = c->n_cor;
  L.row = c->d_cor_row;
  L.ptr = c->d_cor_ptr;
  L.col = c->d_cor_col;
  return L;
}

// The edge rows of w from the Neumann condition, in FP64 (a correction
// computed in FP32 satisfies it only to FP32 rounding of the correction).
static void neumann_w(ufe_ctx *ctx) {
  if (ctx->n_neu) k_neumann_edges<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), ctx->d_pair[0], nullptr);
  k_neumann_scalar_pair_corners<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), ctx->d_pair[0]);
}

static hipEvent_t prof_event(ufe_ctx *ctx) {
  if (ctx->ev_pool.empty()) {
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
  }
  hipEvent_t e = ctx->ev_pool.back();
  ctx->ev_pool.pop_back();
  return e;
}
// Launch one colour kernel; with profiling on, the start/stop events ride on
// the dispatch itself (hipExtLaunchKernelGGL), so they time the kernel's own
// execution and not the queueing around it.
extern "C++" template <typename K, typename... Args>
static void timed_kernel_lds(ufe_ctx *ctx, double bytes, int64_t rows, K kernel, dim3 grid, dim3 block, size_t lds,
                             Args... args) {
  hipEvent_t a = nullptr, b = nullptr;
  // events ride on every PROF_EVERY-th launch: the sample's mean duration is
  // the kernel's, without an event pair on every launch of the timed region
  if (ctx->prof) ctx->prof_acc.total_launches++;
  if (ctx->prof && (ctx->prof_count++ % PROF_EVERY) == 0) {
    a = prof_event(ctx);
    b = prof_event(ctx);
    if (!a || !b) {
      if (a) ctx->ev_pool.push_back(a);
      if (b) ctx->ev_pool.push_back(b);
      a = b = nullptr;
    }
  }
  if (!a) {
    hipLaunchKernelGGL(kernel, grid, block, lds, ctx->stream, args...);
    return;
  }
  hipExtLaunchKernelGGL(kernel, grid, block, lds, ctx->stream, a, b, 0, args...);
  ctx->pending.push_back({a, b, bytes, rows});
}
extern "C++" template <typename K, typename... Args>
static void timed_kernel(ufe_ctx *ctx, double bytes, int64_t rows, K kernel, dim3 grid, dim3 block, Args... args) {
  timed_kernel_lds(ctx, bytes, rows, kernel, grid, block, 0, args...);
}
// after a stream synchronisation: fold the recorded pairs into the profile
static void prof_collect(ufe_ctx *ctx) {
  for (auto &p : ctx->pending) {
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
      ctx->prof_acc.launches++;
      ctx->prof_acc.seconds += ms * 1e-3;
      ctx->prof_acc.algorithmic_bytes += p.bytes;
      ctx->prof_acc.rows += p.rows;
    }
    ctx->ev_pool.push_back(p.a);
    ctx->ev_pool.push_back(p.b);
  }
  ctx->pending.clear();
}

static void enqueue_sweep_fp64(ufe_ctx *ctx, const AaAcMesh &m, double omega, double tol, int max_sweeps,
                               bool with_flags = true) {
  SorFlags *fl = with_flags ? ctx->d_flags : nullptr;
  for (int c = 0; c < 5; c++) {
    const int n = ctx->colour_active[c];
    if (n == 0) continue;
    timed_kernel(ctx, ctx->bytes64[c], n, k_sor_colour, dim3(xcd_grid(n)), dim3(BLOCK), m, ctx->d_pair[0],
                 (const double2 *)ctx->d_pair[1], (const double2 *)ctx->d_pair[2], ctx->colour_start[c], n, omega,
                 fl, (const uint8_t *)(ctx->gl_active ? ctx->d_skip : nullptr));
  }
  if (ctx->n_neu) k_neumann_edges<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), ctx->d_pair[0], fl);
  if (with_flags)
    k_sor_finalize<<<1, 64, 0, ctx->stream>>>(cor_list(ctx), ctx->d_pair[0], ctx->d_flags, tol, max_sweeps);
  else
    k_neumann_scalar_pair_corners<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), ctx->d_pair[0]);
}

// One FP32 colour pass with the tuned launch shape (threads per block, block
// order, load variant), timed like the fixed-shape passes.
extern "C++" template <int BS, int SCHED, int LOADS>
static void launch_sor_f32_shape(ufe_ctx *ctx, const AaAcMesh &m, const Mesh32 &q, float2 *D, const float2 *R, int c,
                                 float omega) {
  const int n = ctx->colour_active[c];
  int g = (n + BS - 1) / BS;
  if (SCHED == 0) g = (g + 7) / 8 * 8;
  timed_kernel(ctx, ctx->bytes32[c], n, k_sor_colour_f32_tuned<BS, SCHED, LOADS>, dim3(g), dim3(BS), m, q, D, R,
               ctx->colour_start[c], n, omega);
}
static void launch_sor_f32(ufe_ctx *ctx, int bs, int sched, int loads, const AaAcMesh &m, const Mesh32 &q, float2 *D,
                           const float2 *R, int c, float omega) {
  switch (bs * 8 + sched * 4 + loads) {
    case 512: launch_sor_f32_shape<64, 0, 0>(ctx, m, q, D, R, c, omega); break;
    case 513: launch_sor_f32_shape<64, 0, 1>(ctx, m, q, D, R, c, omega); break;
    case 514: launch_sor_f32_shape<64, 0, 2>(ctx, m, q, D, R, c, omega); break;
    case 515: launch_sor_f32_shape<64, 0, 3>(ctx, m, q, D, R, c, omega); break;
    case 516: launch_sor_f32_shape<64, 1, 0>(ctx, m, q, D, R, c, omega); break;
    case 517: launch_sor_f32_shape<64, 1, 1>(ctx, m, q, D, R, c, omega); break;
    case 518: launch_sor_f32_shape<64, 1, 2>(ctx, m, q, D, R, c, omega); break;
    case 519: launch_sor_f32_shape<64, 1, 3>(ctx, m, q, D, R, c, omega); break;
    case 1024: launch_sor_f32_shape<128, 0, 0>(ctx, m, q, D, R, c, omega); break;
    case 1025: launch_sor_f32_shape<128, 0, 1>(ctx, m, q, D, R, c, omega); break;
    case 1026: launch_sor_f32_shape<128, 0, 2>(ctx, m, q, D, R, c, omega); break;
    case 1027: launch_sor_f32_shape<128, 0, 3>(ctx, m, q, D, R, c, omega); break;
    case 1028: launch_sor_f32_shape<128, 1, 0>(ctx, m, q, D, R, c, omega); break;
    case 1029: launch_sor_f32_shape<128, 1, 1>(ctx, m, q, D, R, c, omega); break;
    case 1030: launch_sor_f32_shape<128, 1, 2>(ctx, m, q, D, R, c, omega); break;
    case 1031: launch_sor_f32_shape<128, 1, 3>(ctx, m, q, D, R, c, omega); break;
    case 2048: launch_sor_f32_shape<256, 0, 0>(ctx, m, q, D, R, c, omega); break;
    case 2049: launch_sor_f32_shape<256, 0, 1>(ctx, m, q, D, R, c, omega); break;
    case 2050: launch_sor_f32_shape<256, 0, 2>(ctx, m, q, D, R, c, omega); break;
    case 2051: launch_sor_f32_shape<256, 0, 3>(ctx, m, q, D, R, c, omega); break;
    case 2052: launch_sor_f32_shape<256, 1, 0>(ctx, m, q, D, R, c, omega); break;
    case 2053: launch_sor_f32_shape<256, 1, 1>(ctx, m, q, D, R, c, omega); break;
    case 2054: launch_sor_f32_shape<256, 1, 2>(ctx, m, q, D, R, c, omega); break;
    case 2055: launch_sor_f32_shape<256, 1, 3>(ctx, m, q, D, R, c, omega); break;
    case 4096: launch_sor_f32_shape<512, 0, 0>(ctx, m, q, D, R, c, omega); break;
    case 4097: launch_sor_f32_shape<512, 0, 1>(ctx, m, q, D, R, c, omega); break;
    case 4098: launch_sor_f32_shape<512, 0, 2>(ctx, m, q, D, R, c, omega); break;
    case 4099: launch_sor_f32_shape<512, 0, 3>(ctx, m, q, D, R, c, omega); break;
    case 4100: launch_sor_f32_shape<512, 1, 0>(ctx, m, q, D, R, c, omega); break;
    case 4101: launch_sor_f32_shape<512, 1, 1>(ctx, m, q, D, R, c, omega); break;
    case 4102: launch_sor_f32_shape<512, 1, 2>(ctx, m, q, D, R, c, omega); break;
    case 4103: launch_sor_f32_shape<512, 1, 3>(ctx, m, q, D, R, c, omega); break;
    default: launch_sor_f32_shape<256, 0, 0>(ctx, m, q, D, R, c, omega); break;
  }
}

// The Neumann update of an FP32 pair vector: the edge rows, then the corners.
// (One workgroup doing both, with a barrier between, took 11.2 us at 1M against
// 4.7 + 4.7 us for the two kernels.)
static void neumann_f32(ufe_ctx *ctx, float2 *D) {
  if (ctx->n_neu) k_neumann_edges_f32<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), D);
  k_neumann_corners_f32<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), D);
}

// skip_first: leave out the first colour of the pass (a preconditioner that
// alternates direction would otherwise repeat the previous pass's last colour
// with nothing changed in between).  from_zero: the sweep starts from D = 0
// whatever D holds: one kernel zeroes D and updates the first colour's rows,
// which need neither neighbours nor coefficients (k_sor_zero_colour_f32).
static void enqueue_sweep_fp32(ufe_ctx *ctx, const AaAcMesh &m, float omega, float2 *D = nullptr,
                               const float2 *R = nullptr, bool backward = false, bool skip_first = false,
                               bool neumann = true, bool from_zero = false) {
  Mesh32 q;
  q.cU = ctx->d_cU32;
  q.Sxy = ctx->d_Sxy32;
  q.EV = ctx->d_EV32;
  q.skip = ctx->gl_active ? ctx->d_skip : nullptr;
  if (!D) D = ctx->d_D32;
  if (!R) R = ctx->d_R32;
  if (from_zero) {
    const int c = backward ? 4 : 0;
    k_sor_zero_colour_f32<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(
        ctx->nA, q.EV, R, q.skip, D, ctx->colour_start[c], skip_first ? 0 : ctx->colour_active[c], omega);
  }
  for (int k = skip_first || from_zero ? 1 : 0; k < 5; k++) {
    const int c = backward ? 4 - k : k;
    const int n = ctx->colour_active[c];
    if (n == 0) continue;
    launch_sor_f32(ctx, ctx->tune_bs, ctx->tune_sched, ctx->tune_loads, m, q, D, R, c, omega);
  }
  if (!neumann) return;
  neumann_f32(ctx, D);
}

// FP64 sweep on an arbitrary vector pair (Krylov preconditioner)
static void enqueue_sweep_fp64_vec(ufe_ctx *ctx, const AaAcMesh &m, double omega, double2 *D, const double2 *R,
                                   bool backward, bool skip_first = false, bool neumann = true) {
  for (int k = skip_first ? 1 : 0; k < 5; k++) {
    const int c = backward ? 4 - k : k;
    const int n = ctx->colour_active[c];
    if (n == 0) continue;
    timed_kernel(ctx, ctx->bytes64[c], n, k_sor_colour, dim3(xcd_grid(n)), dim3(BLOCK), m, D,
                 (const double2 *)ctx->d_pair[1], R, ctx->colour_start[c], n, omega, (SorFlags *)nullptr,
                 (const uint8_t *)(ctx->gl_active ? ctx->d_skip : nullptr));
  }
  if (!neumann) return;
  if (ctx->n_neu) k_neumann_edges<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), D, nullptr);
  k_neumann_scalar_pair_corners<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), D);
}

// ---------------------------------------------------------------------------
// Aggregation multigrid preconditioner for the FP32 correction solve: set-up
// on the host once per mesh (the off-diagonal coefficients depend on the mesh
// only), the diagonal pairs of every level rebuilt on the device with each
// new system, and one K-cycle per application.
// ---------------------------------------------------------------------------
static ActiveRanges active_ranges(ufe_ctx *ctx);

constexpr int AMG_KSTEP_MIN = 1000;      // levels with at least this many points take two cycles
constexpr float AMG_BJ_OMEGA = 0.8f;     // damping of the coarse-level block Jacobi
constexpr int AMG_COARSE_SWEEPS = 20;    // coarsest level too large for the dense inverse
constexpr size_t AMG_TAIL_LDS_MARGIN = 256;     // bytes of LDS left unused by k_amg_tail
constexpr int AMG_FUSE_MAX_POINTS = 1 << 24;   // levels up to this size take the fused cycle kernels
constexpr size_t AMG_FUSE_LDS_MAX = 56 * 1024;  // their LDS arrays (36 bytes per listed point; 6 KiB static beside)
constexpr size_t AMG_FUSE_LDS_HELD = 58 * 1024; // and with the rows: 64 KiB less the static part

// Coarse levels of at most this many points get the fused kernels' blocks and
// halos when their block lists fit in LDS (UFE_AMG_FUSE_MAX=n sets the size
// limit); their K-step dots follow those blocks whether the cycle steps run
// fused or, with UFE_AMG_FUSE=0 in the environment at set-up, one kernel each.
static bool amg_fuse_on() {
  const char *off = std::getenv("UFE_AMG_FUSE");
  return !(off && off[0] == '0');
}
// Deepest halo to build (UFE_AMG_FUSE_DEPTH=1..3 in the environment at set-up
// lowers it; a level whose lists do not fit in LDS takes a shallower one).
static int amg_fuse_depth() {
  const char *env = std::getenv("UFE_AMG_FUSE_DEPTH");
  if (env && env[0]) {
    const long v = std::strtol(env, nullptr, 10);
    if (v >= 1 && v <= AMG_FUSE_NU) return (int)v;
  }
  return AMG_FUSE_NU;
}
// Most points a fused-kernel block owns on coarse level l (1-based) of n
// points: the largest power of two up to n / 512, within 32..AMG_FUSE_BLOCK,
// so that a level has about 512 blocks or more (two per CU) unless its blocks
// are already small.  The coarse levels' kernels are bound by their dependent
// steps, and a block's steps take fewer rounds of its threads when it lists
// fewer points; the halo work this repeats is cheap on those levels.  The l-th
// entry of UFE_AMG_FUSE_OWN (a comma list, its last entry repeated; each
// 16..AMG_FUSE_BLOCK) overrides it.  Only the order of the K-step dots' partial
// sums depends on the blocks.
static int amg_fuse_own(int l, int n) {
  int v = 32;
  while (v < AMG_FUSE_BLOCK && 2 * v <= n / 512) v *= 2;
  const char *env = std::getenv("UFE_AMG_FUSE_OWN");
  if (env && env[0]) {
    const char *s = env;
    for (int k = 1; k <= l && *s; k++) {
      char *end = nullptr;
      const long x = std::strtol(s, &end, 10);
      if (end == s) break;
      if (x >= 16 && x <= AMG_FUSE_BLOCK) v = (int)x;
      s = *end == ',' ? end + 1 : end;
    }
  }
  return v;
}
// A fused level's second K-step cycle finishes step 1 in its pre-smoothing
// kernel, every block summing the step-1 partials itself, when the level has
// at most this many partials; larger levels keep the finisher kernels, where
// the sums would cost each of the many blocks more than the launch they save
// (UFE_AMG_KFOLD_MAX=n in the environment at set-up sets the limit, 0 turns
// the folding off).
constexpr int AMG_KFOLD_MAX_PARTS = 1024;
static int amg_kfold_max() {
  const char *env = std::getenv("UFE_AMG_KFOLD_MAX");
  if (env && env[0]) {
    const long v = std::strtol(env, nullptr, 10);
    if (v >= 0 && v < (1L << 30)) return (int)v;
  }
  return AMG_KFOLD_MAX_PARTS;
}
static int amg_fuse_max() {
  const char *env = std::getenv("UFE_AMG_FUSE_MAX");
  if (env && env[0]) {
    const long v = std::strtol(env, nullptr, 10);
    if (v >= 0 && v < (1L << 30)) return (int)v;
  }
  return AMG_FUSE_MAX_POINTS;
}

// Dynamic LDS that k_amg_tail may take on this device: the device's limit per
// workgroup (160 KiB on gfx950) less the kernel's static LDS.
static int amg_tail_lds_budget(ufe_ctx *ctx, size_t *out) {
  int per_block = 0;
  HIPCHK(ctx, hipDeviceGetAttribute(&per_block, hipDeviceAttributeMaxSharedMemoryPerBlock, ctx->device));
  size_t stat = 0;
  const void *kernels[2] = {reinterpret_cast<const void *>(&k_amg_tail<true>),
                            reinterpret_cast<const void *>(&k_amg_tail<false>)};
  for (const void *k : kernels) {
    hipFuncAttributes fa{};
    HIPCHK(ctx, hipFuncGetAttributes(&fa, k));
    stat = std::max(stat, (size_t)fa.sharedSizeBytes + AMG_TAIL_LDS_MARGIN);
  }
  *out = (size_t)per_block > stat ? (size_t)per_block - stat : 0;
  if (*out + stat > 65536) {
    for (const void *k : kernels)
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)*out) != hipSuccess) {
        (void)hipGetLastError();     // the runtime keeps the 64 KiB default
        *out = 65536 > stat ? 65536 - stat : 0;
        break;
      }
  }
  return UFE_OK;
}

// Levels with at least this many points take K-steps (UFE_AMG_KSTEP_MIN in the
// environment at set-up overrides AMG_KSTEP_MIN).
static int amg_kstep_min() {
  const char *env = std::getenv("UFE_AMG_KSTEP_MIN");
  if (env && env[0]) {
    const long v = std::strtol(env, nullptr, 10);
    if (v > 0 && v < (1L << 30)) return (int)v;
  }
  return AMG_KSTEP_MIN;
}
constexpr int AMG_MAX_LEVELS = 16;

// The small-level kernel's images (see AmgTail): the constant arrays of the
// tail levels packed in its LDS layout, when they fit beside the vectors.  The
// diagonal pairs are written into image B by k_amg_ev with every new system.
static int amg_tail_images(ufe_ctx *ctx) {
  ctx->amg_tail_imgA = ctx->amg_tail_imgAT = ctx->amg_tail_imgB = nullptr;
  ctx->amg_tail_wA = ctx->amg_tail_wB = 0;
  const int l0 = ctx->amg_tail_l0, L = (int)ctx->amg.size();
  const char *env = std::getenv("UFE_AMG_TAIL_IMAGES");   // 0: read the arrays from global memory
  if (l0 <= 0 || (env && env[0] == '0')) return UFE_OK;
  size_t vec = 0, bA = 0, bB = 0;
  for (int k = 0; k < L - l0; k++) {
    const AmgLevel &V = ctx->amg[l0 + k];
    vec += 3 * (size_t)V.n * sizeof(float2);
    ctx->amg_tail_offA[k] = (int)bA;
    ctx->amg_tail_offB[k] = (int)bB;
    bA += amg_tail_bytes_A(V.n, (int)V.nnz);
    bB += amg_tail_bytes_B(V.n, V.nmem, V.nagg, k > 0);
  }
  vec = (vec + 15) & ~(size_t)15;
  if (vec + bA + bB > ctx->amg_tail_lds) return UFE_OK;
  int r;
  if ((r = dalloc(ctx, &ctx->amg_tail_imgA, bA / 16))) return r;
  if ((r = dalloc(ctx, &ctx->amg_tail_imgAT, bA / 16))) return r;
  if ((r = dalloc(ctx, &ctx->amg_tail_imgB, bB / 16))) return r;
  auto put = [&](uint4 *img, size_t off, const void *src, size_t bytes) -> int {
    if (bytes)
      HIPCHK(ctx, hipMemcpyAsync(reinterpret_cast<char *>(img) + off, src, bytes, hipMemcpyDeviceToDevice,
                                 ctx->stream));
    return UFE_OK;
  };
  for (int k = 0; k < L - l0; k++) {
    AmgLevel &V = ctx->amg[l0 + k];
    const size_t n = (size_t)V.n, nnz = (size_t)V.nnz, a = ctx->amg_tail_offA[k], b = ctx->amg_tail_offB[k];
    if ((r = put(ctx->amg_tail_imgA, a, V.cf, nnz * 8)) || (r = put(ctx->amg_tail_imgA, a + nnz * 8, V.col, nnz * 4)) ||
        (r = put(ctx->amg_tail_imgA, a + nnz * 12, V.ptr, (n + 1) * 4)) ||
        (r = put(ctx->amg_tail_imgAT, a, V.cfT, nnz * 8)) || (r = put(ctx->amg_tail_imgAT, a + nnz * 8, V.colT, nnz * 4)) ||
        (r = put(ctx->amg_tail_imgAT, a + nnz * 12, V.ptrT, (n + 1) * 4)) ||
        (r = put(ctx->amg_tail_imgB, b + n * 8, V.S, n * 4)))
      return r;
    if (k > 0 && ((r = put(ctx->amg_tail_imgB, b + n * 12, V.mptr, (n + 1) * 4)) ||
                  (r = put(ctx->amg_tail_imgB, b + n * 12 + (n + 1) * 4, V.mem, (size_t)V.nmem * 4)) ||
                  (r = put(ctx->amg_tail_imgB, b + n * 12 + (n + 1 + V.nmem) * 4, V.agg, (size_t)V.nagg * 4))))
      return r;
    V.ev32_img = reinterpret_cast<float2 *>(reinterpret_cast<char *>(ctx->amg_tail_imgB) + b);
  }
  ctx->amg_tail_wA = (int)(bA / 16);
  ctx->amg_tail_wB = (int)(bB / 16);
  return UFE_OK;
}

// The colour-ordered neighbour lists on the host, read back once for the multigrid
// set-up and the patches (empty: not read)
struct HostLists {
  std::vector<int64_t> cptr;
  std::vector<uint8_t> deg;
  std::vector<int32_t> col, nrow, nptr, ncol, crow, cptr2, ccol;   // neighbours; edge points; corners
};
static int host_lists(ufe_ctx *ctx, HostLists &L) {
  if (!L.cptr.empty()) return UFE_OK;
  const int nA = ctx->nA, nchunk = (nA + SELL - 1) / SELL;
  int r;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  auto get_list = [&](int n, const int32_t *drow, const int32_t *dptr, const int32_t *dcol,
                      std::vector<int32_t> &row, std::vector<int32_t> &ptr, std::vector<int32_t> &cl) -> int {
    row.resize(n);
    ptr.assign(n + 1, 0);
    if (n == 0) return UFE_OK;
    HIPCHK(ctx, hipMemcpy(row.data(), drow, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    HIPCHK(ctx, hipMemcpy(ptr.data(), dptr, sizeof(int32_t) * (n + 1), hipMemcpyDeviceToHost));
    cl.resize(ptr[n]);
    HIPCHK(ctx, hipMemcpy(cl.data(), dcol, sizeof(int32_t) * ptr[n], hipMemcpyDeviceToHost));
    return UFE_OK;
  };
  if ((r = get_list(ctx->n_neu, ctx->d_neu_row, ctx->d_neu_ptr, ctx->d_neu_col, L.nrow, L.nptr, L.ncol))) return r;
  if ((r = get_list(ctx->n_cor, ctx->d_cor_row, ctx->d_cor_ptr, ctx->d_cor_col, L.crow, L.cptr2, L.ccol))) return r;
  L.deg.resize(nA);
  HIPCHK(ctx, hipMemcpy(L.deg.data(), ctx->d_deg, nA, hipMemcpyDeviceToHost));
  std::vector<int64_t> cptr(nchunk + 1);
  HIPCHK(ctx, hipMemcpy(cptr.data(), ctx->d_chunk_ptr, sizeof(int64_t) * (nchunk + 1), hipMemcpyDeviceToHost));
  L.col.resize(cptr[nchunk]);
  HIPCHK(ctx, hipMemcpy(L.col.data(), ctx->d_col, sizeof(int32_t) * L.col.size(), hipMemcpyDeviceToHost));
  L.cptr = std::move(cptr);          // last: marks the lists as read
  return UFE_OK;
}

static int amg_setup(ufe_ctx *ctx, HostLists &H) {
  if (ctx->amg_ready) return UFE_OK;
  const auto t0 = std::chrono::steady_clock::now();
  const int nA = ctx->nA;
  int r;
  // the fine operator, read back from the device
  if ((r = host_lists(ctx, H))) return r;
  const std::vector<int64_t> &cptr = H.cptr;
  const std::vector<uint8_t> &deg = H.deg;
  const std::vector<int32_t> &col = H.col, &nrow = H.nrow, &nptr = H.nptr, &ncol = H.ncol, &crow = H.crow,
                             &cptr2 = H.cptr2, &ccol = H.ccol;
  const int64_t ne = (int64_t)col.size();
  std::vector<double2> cU(ne);
  std::vector<double> Sxy(nA);
  HIPCHK(ctx, hipMemcpy(cU.data(), ctx->d_cU, sizeof(double2) * ne, hipMemcpyDeviceToHost));
  HIPCHK(ctx, hipMemcpy(Sxy.data(), ctx->d_Sxy, sizeof(double) * nA, hipMemcpyDeviceToHost));
  // fine points: the SOR rows in colour order
  std::vector<int32_t> pid(nA, -1), rows;
  for (int c = 0; c < 5; c++)
    for (int p = ctx->colour_start[c]; p < ctx->colour_start[c] + ctx->colour_active[c]; p++) {
      pid[p] = (int32_t)rows.size();
      rows.push_back(p);
    }
  const int n0 = (int)rows.size();
  if (n0 == 0) {
    ctx->err = "no SOR rows to aggregate";
    return UFE_BAD_INPUT;
  }
  // the Neumann rows as weighted sums of fine points, then the operator on the
  // fine points with them eliminated
  std::vector<int32_t> exi;
  std::vector<AmgExpansion> exl;
  amg_neumann_expansions(pid, nrow, nptr, ncol, crow, cptr2, ccol, exi, exl);
  static_assert(sizeof(AmgPair) == sizeof(double2), "AmgPair must have the layout of double2");
  std::vector<AmgHostOp> ops(1);
  amg_fine_operator(rows, SELL, cptr, deg, col, reinterpret_cast<const AmgPair *>(cU.data()), Sxy, pid, exi, exl,
                    ops[0]);
  // coarsen until the dense inverse fits (at least one coarse level)
  std::vector<std::vector<int32_t>> aggs, mptrs, mems;
  std::vector<std::vector<AmgPair>> intras;
  while ((int)ops.size() < AMG_MAX_LEVELS && (ops.size() == 1 || ops.back().n > AMG_DIRECT)) {
    int na = 0;
    std::vector<int32_t> agg = amg_aggregate(ops.back(), &na);
    if (ops.size() > 1 && na > (int)(0.85 * ops.back().n)) break;   // coarsening stalled
    AmgHostOp C;
    std::vector<int32_t> mptr, mem;
    std::vector<AmgPair> intra;
    amg_galerkin(ops.back(), agg, na, C, mptr, mem, intra);
    intras.push_back(std::move(intra));
    aggs.push_back(std::move(agg));
    mptrs.push_back(std::move(mptr));
    mems.push_back(std::move(mem));
    ops.push_back(std::move(C));
  }
  const int L = (int)ops.size();
  const int kstep_min = amg_kstep_min();
  const int fuse_max = amg_fuse_max();
  const bool fuse_on = amg_fuse_on();
  ctx->amg_kfold_max = amg_kfold_max();
  if ((r = amg_tail_lds_budget(ctx, &ctx->amg_tail_lds))) return r;
  ctx->amg.assign(L, AmgLevel{});
  ctx->amg[0].n = n0;
  for (int l = 1; l < L; l++) {
    AmgLevel &V = ctx->amg[l];
    const AmgHostOp &C = ops[l];
    V.n = C.n;
    V.nnz = (int64_t)C.col.size();
    V.kstep = l < L - 1 && C.n >= kstep_min;
    std::vector<float2> cf32(std::max<size_t>(C.cf.size(), 1));
    for (size_t k = 0; k < C.cf.size(); k++) cf32[k] = make_float2((float)C.cf[k].x, (float)C.cf[k].y);
    std::vector<float> S32(C.n);
    for (int i = 0; i < C.n; i++) S32[i] = (float)C.S[i];
    std::vector<int32_t> colv = C.col;
    if (colv.empty()) colv.push_back(0);
    if ((r = dupload(ctx, &V.ptr, C.ptr.data(), C.ptr.size()))) return r;
    if ((r = dupload(ctx, &V.col, colv.data(), colv.size()))) return r;
    if ((r = dupload(ctx, &V.cf, cf32.data(), cf32.size()))) return r;
    std::vector<int32_t> pT, cT;   // the transposed couplings (adjoint solves)
    std::vector<float2> fT;
    {
      amg_transpose(C.n, C.ptr, C.col, cf32, pT, cT, fT);
      if (cT.empty()) {
        cT.push_back(0);
        fT.push_back(make_float2(0.0f, 0.0f));
      }
      if ((r = dupload(ctx, &V.ptrT, pT.data(), pT.size()))) return r;
      if ((r = dupload(ctx, &V.colT, cT.data(), cT.size()))) return r;
      if ((r = dupload(ctx, &V.cfT, fT.data(), fT.size()))) return r;
    }
    if ((r = dupload(ctx, &V.S, S32.data(), S32.size()))) return r;
    if (l < L - 1 && C.n <= fuse_max) {   // the fused cycle kernels' blocks and halos, as deep as fit
      std::vector<int32_t> gptr, gagg;
      amg_blocks_by_aggregates(ops[l + 1].n, ops[l + 1].ptr, ops[l + 1].col, mptrs[l], amg_fuse_own(l, C.n), gptr, gagg);
      AmgHalos H;
      for (int depth = amg_fuse_depth(); depth >= 1; depth--) {
        amg_block_halos(C.n, C.ptr, C.col, gptr, gagg, mptrs[l], mems[l], depth, H, &pT, &cT);
        if ((size_t)H.max_ext * 36 <= AMG_FUSE_LDS_MAX) break;
      }
      if ((size_t)H.max_ext * 36 <= AMG_FUSE_LDS_MAX) {
        std::vector<float2> lcf(std::max<size_t>(H.lsrc.size(), 1));
        for (size_t k = 0; k < H.lsrc.size(); k++) lcf[k] = cf32[H.lsrc[k]];
        if (H.lcol.empty()) H.lcol.push_back(0);
        // local columns index lists of at most max_ext points: 16 bits hold them
        static_assert(AMG_FUSE_LDS_MAX / 36 < 65536, "local columns must fit in 16 bits");
        const std::vector<uint16_t> lcol16(H.lcol.begin(), H.lcol.end());
        int32_t *d_ext_ptr, *d_ext, *d_cnt, *d_rstart, *d_rptr, *d_gptr, *d_gagg, *d_glo;
        uint16_t *d_lcol;
        float2 *d_lcf;
        if ((r = dupload(ctx, &d_ext_ptr, H.ext_ptr.data(), H.ext_ptr.size())) ||
            (r = dupload(ctx, &d_ext, H.ext.data(), H.ext.size())) ||
            (r = dupload(ctx, &d_cnt, H.cnt.data(), H.cnt.size())) ||
            (r = dupload(ctx, &d_rstart, H.rstart.data(), H.rstart.size())) ||
            (r = dupload(ctx, &d_rptr, H.rptr.data(), H.rptr.size())) ||
            (r = dupload(ctx, &d_lcol, lcol16.data(), lcol16.size())) ||
            (r = dupload(ctx, &d_lcf, lcf.data(), lcf.size())) ||
            (r = dupload(ctx, &d_gptr, H.gptr.data(), H.gptr.size())) ||
            (r = dupload(ctx, &d_gagg, H.gagg.data(), H.gagg.size())) ||
            (r = dupload(ctx, &d_glo, H.glo.data(), H.glo.size())))
          return r;
        V.F = AmgFuse{H.depth, d_ext_ptr, d_ext, d_cnt, d_rstart, d_rptr, d_lcol, d_lcf, V.S, nullptr,
                      d_gptr, d_gagg, d_glo, H.max_ext, 0, 0};
        // the blocks' rows beside the lists where both orientations fit
        int nnz = 0, rows = 0;
        for (int b = 0; b < H.nblocks; b++) {
          const int q0 = H.rstart[b], q1 = H.rstart[b + 1];
          rows = std::max(rows, q1 - q0);
          nnz = std::max(nnz, H.rptr[q1] - H.rptr[q0]);
          if (H.transposed_ok) nnz = std::max(nnz, H.rptrT[q1] - H.rptrT[q0]);
        }
        V.F.nnz_cap = nnz;
        V.F.row_cap = rows;
        if (amg_fuse_lds(V.F) > AMG_FUSE_LDS_HELD) V.F.nnz_cap = V.F.row_cap = 0;
        V.fuse_blocks = H.nblocks;
        V.blocks = true;
        V.fuse = fuse_on;
        if (H.transposed_ok) {   // the same blocks for the transposed hierarchy
          std::vector<float2> lcfT(std::max<size_t>(H.lsrcT.size(), 1));
          for (size_t k = 0; k < H.lsrcT.size(); k++) lcfT[k] = fT[H.lsrcT[k]];
          if (H.lcolT.empty()) H.lcolT.push_back(0);
          const std::vector<uint16_t> lcolT16(H.lcolT.begin(), H.lcolT.end());
          if ((r = dupload(ctx, &V.fuse_rptrT, H.rptrT.data(), H.rptrT.size())) ||
              (r = dupload(ctx, &V.fuse_lcolT, lcolT16.data(), lcolT16.size())) ||
              (r = dupload(ctx, &V.fuse_lcfT, lcfT.data(), lcfT.size())))
            return r;
          V.fuseT = true;
        }
      }
    }
    // the part of the diagonal that does not come from the level above: at level
    // 1 the fine fixed parts (Neumann self-couplings) as well, since the fine
    // diagonal pairs EV do not hold them; below, the couplings inside each
    // aggregate only (the members' diagonals already hold their fixed parts)
    const std::vector<AmgPair> &own = l == 1 ? C.fd : intras[l - 1];
    if ((r = dupload(ctx, &V.fd, reinterpret_cast<const double2 *>(own.data()), own.size()))) return r;
    if ((r = dalloc(ctx, &V.ev64, (size_t)C.n))) return r;
    if ((r = dalloc(ctx, &V.ev32, (size_t)C.n))) return r;
    V.F.ev = V.ev32;
    // members and aggregate map: level 1 in fine rows, deeper levels in points
    std::vector<int32_t> mem = mems[l - 1];
    std::vector<int32_t> agg;
    if (l == 1) {
      for (auto &i : mem) i = rows[i];
      agg.assign(nA, -1);
      for (int i = 0; i < n0; i++) agg[rows[i]] = aggs[0][i];
    } else {
      agg = aggs[l - 1];
    }
    if ((r = dupload(ctx, &V.mptr, mptrs[l - 1].data(), mptrs[l - 1].size()))) return r;
    if ((r = dupload(ctx, &V.mem, mem.data(), mem.size()))) return r;
    if ((r = dupload(ctx, &V.agg, agg.data(), agg.size()))) return r;
    V.nmem = (int)mem.size();
    V.nagg = (int)agg.size();
    float2 **vecs[8] = {&V.b, &V.t, &V.e1, &V.e2, &V.w1, &V.w2, &V.rc2, &V.r};
    for (float2 **v : vecs)
      if ((r = dalloc(ctx, v, (size_t)C.n))) return r;
    if ((r = dalloc(ctx, &V.part, (size_t)3 * std::max(AMG_DOT_BLOCKS, V.fuse_blocks)))) return r;
    if ((r = dalloc(ctx, &V.sc, (size_t)8))) return r;
    HIPCHK(ctx, hipMemset(V.sc, 0, 8 * sizeof(double)));
  }
  if ((r = dalloc(ctx, &ctx->amg_y, (size_t)nA))) return r;
  if ((r = dalloc(ctx, &ctx->amg_y64, (size_t)nA))) return r;
  if ((r = dalloc(ctx, &ctx->amg_v32, (size_t)nA))) return r;
  if ((r = dalloc(ctx, &ctx->amg_z32, (size_t)nA))) return r;
  AmgLevel &Lc = ctx->amg[L - 1];
  ctx->amg_direct = Lc.n <= AMG_DIRECT;
  if (ctx->amg_direct) {
    const AmgHostOp &C = ops[L - 1];
    std::vector<AmgPair> cf = C.cf;
    if (cf.empty()) cf.push_back(AmgPair{0.0, 0.0});
    if ((r = dupload(ctx, &Lc.cf64, reinterpret_cast<const double2 *>(cf.data()), cf.size()))) return r;
    if ((r = dupload(ctx, &Lc.S64, C.S.data(), C.S.size()))) return r;
    const size_t N = 2 * (size_t)Lc.n;
    if ((r = dalloc(ctx, &ctx->amg_inv, 2 * N * N))) return r;   // the inverse and its transpose
    if (N * N * sizeof(double) > 65536)                           // the matrix in LDS
      HIPCHK(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(&k_amg_dense_inv),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)(N * N * sizeof(double))));
  }
  HIPCHK(ctx, hipDeviceSynchronize());
  // The levels below the last K-step level, each visited by one V-cycle, are
  // solved by one workgroup per visit (k_amg_tail) when their vectors fit in
  // LDS; UFE_AMG_TAIL=0 in the environment keeps one kernel per step.
  ctx->amg_tail_l0 = 0;
  {
    const char *env = std::getenv("UFE_AMG_TAIL");
    int l0 = L - 1;
    while (l0 > 1 && !ctx->amg[l0 - 1].kstep) l0--;
    size_t lds = 0;
    for (int l = l0; l < L; l++) lds += 3 * (size_t)ctx->amg[l].n * sizeof(float2);
    const int nlev = L - l0;
    if (!(env && env[0] == '0') && nlev >= 2 && nlev <= AMG_TAIL_LEVELS && lds <= ctx->amg_tail_lds)
      ctx->amg_tail_l0 = l0;
  }
  if ((r = amg_tail_images(ctx))) return r;
  ctx->amg_ready = true;
  ctx->amg_setup_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return UFE_OK;
}

static AmgOp amg_op(const ufe_ctx *ctx, const AmgLevel &V) {
  AmgOp A;
  A.n = V.n;
  A.ptr = ctx->amg_T ? V.ptrT : V.ptr;
  A.col = ctx->amg_T ? V.colT : V.col;
  A.cf = ctx->amg_T ? V.cfT : V.cf;
  A.S = V.S;
  A.ev = V.ev32;
  return A;
}

// the diagonal pairs of every level for the current system (FP64 EV in d_pair[1])
static void amg_refresh(ufe_ctx *ctx) {
  const int L = (int)ctx->amg.size();
  for (int l = 1; l < L; l++) {
    AmgLevel &V = ctx->amg[l];
    const double2 *evf = l == 1 ? ctx->d_pair[1] : ctx->amg[l - 1].ev64;
    k_amg_ev<<<nblk(V.n), BLOCK, 0, ctx->stream>>>(V.n, V.mptr, V.mem, evf, V.fd, V.ev64, V.ev32, V.ev32_img);
  }
  if (ctx->amg_direct) {
    AmgLevel &V = ctx->amg[L - 1];
    const size_t lds = 4 * (size_t)V.n * V.n * sizeof(double);
    k_amg_dense_inv<<<1, AMG_INV_THREADS, lds, ctx->stream>>>(V.n, V.ptr, V.col, V.cf64, V.S64, V.ev64, ctx->amg_inv);
  }
}

static void amg_solve_level(ufe_ctx *ctx, int l);

// level l's cycle runs as k_amg_fuse_pre / k_amg_fuse_post (halos deep enough
// for the smoothing, local rows of the operator in use)
static bool amg_fused_cycle(const ufe_ctx *ctx, int l) {
  const AmgLevel &V = ctx->amg[l];
  return l >= 1 && V.fuse && (!ctx->amg_T || V.fuseT) && std::max(1, ctx->amg_nu) <= V.F.depth;
}

// K-step partial sums of level V: one per fused-kernel block when it has them
static int amg_dot_count(const AmgLevel &V) {
  return V.blocks ? V.fuse_blocks : std::min(AMG_DOT_BLOCKS, nblk(V.n, 256));
}

// Level 1's step-2 coefficients: added up by every block of the fine prolongation
// up to AMG_LATE_KFIN blocks of it, by a launch of their own (4 us) above, where the
// blocks' reading of the partial sums (6 KB each) takes longer than that
constexpr int AMG_LATE_KFIN = 1024;
static bool amg_late_kfin(const ufe_ctx *ctx) { return nblk(ctx->nA) <= AMG_LATE_KFIN; }
static AmgStep2 amg_fine_step2(const ufe_ctx *ctx) {
  const AmgLevel &C = ctx->amg[1];
  if (!C.kstep) return {nullptr, nullptr, 0};
  if (!amg_late_kfin(ctx)) return {C.sc, nullptr, 0};
  return {C.sc, C.part, amg_dot_count(C)};
}

// The K-step dots of a cycle's result (y = A x, and y.a, y.y, y.c by block),
// which the fused post-smoothing computes itself when its halos reach one ring
// beyond the smoothing; done reports whether it did.
struct AmgDots {
  const float2 *a;                  // null: the cycle's right-hand side
  bool c_rhs;                       // y.c with c the right-hand side
  float2 *y;
  double *part;
  bool done;
};

// The step-1 finish of a K-step (alpha1 from the partials, rc2 = b - alpha1 w1)
// done by the second cycle's fused pre-smoothing kernel (amg_kfold_max).
struct AmgFold {
  const float2 *w1;
  int knb;
  const double *kpart;
  double *sc;
  float2 *rc2;
};

// x ~ A_l^-1 b: nu block-Jacobi sweeps, the coarse correction, nu sweeps.  The
// 2 nu sweeps alternate between t and x, starting in t, so they end in x.  With
// fold given (fused levels only) the right-hand side is fold->rc2, which the
// pre-smoothing kernel forms from b.
static void amg_cycle(ufe_ctx *ctx, int l, const float2 *b, float2 *x, AmgDots *dots = nullptr,
                      const AmgFold *fold = nullptr) {
  AmgLevel &V = ctx->amg[l];
  const AmgOp A = amg_op(ctx, V);
  const int nb = nblk(V.n), last = (int)ctx->amg.size() - 1;
  if (l == last) {
    if (ctx->amg_direct) {
      k_amg_dense_apply<<<1, AMG_DENSE_THREADS, 0, ctx->stream>>>(V.n, ctx->amg_inv, b, x, ctx->amg_T ? 1 : 0);
      return;
    }
    k_amg_bj<<<nb, BLOCK, 0, ctx->stream>>>(A, b, nullptr, V.t, AMG_BJ_OMEGA);
    float2 *src = V.t, *dst = x;
    for (int s = 1; s < 2 * AMG_COARSE_SWEEPS; s++) {
      k_amg_bj<<<nb, BLOCK, 0, ctx->stream>>>(A, b, src, dst, AMG_BJ_OMEGA);
      std::swap(src, dst);
    }
    return;
  }
  const int nu = std::max(1, ctx->amg_nu);
  if (amg_fused_cycle(ctx, l)) {   // two kernels with block halos, same results
    AmgLevel &C = ctx->amg[l + 1];
    const size_t lds = amg_fuse_lds(V.F);
    const bool held = V.F.nnz_cap > 0;
    AmgFuse F = V.F;
    if (ctx->amg_T) {
      F.rptr = V.fuse_rptrT;
      F.lcol = V.fuse_lcolT;
      F.lcf = V.fuse_lcfT;
    }
    // the blocks are whole aggregates of level l + 1: the pre-smoothing kernel
    // also sums their members' residuals into C.b (as k_amg_gather)
    auto pre = held ? k_amg_fuse_pre<true> : k_amg_fuse_pre<false>;
    pre<<<V.fuse_blocks, AMG_FUSE_BLOCK, lds, ctx->stream>>>(
        F, nu, b, V.t, C.b, AMG_BJ_OMEGA, fold ? fold->w1 : nullptr, fold ? fold->knb : 0,
        fold ? fold->kpart : nullptr, fold ? fold->sc : nullptr, fold ? fold->rc2 : nullptr);
    if (fold) b = fold->rc2;
    amg_solve_level(ctx, l + 1);
    // a K-step level below leaves its step-2 partials to this kernel (amg_solve_level)
    const int cnd = amg_dot_count(C);
    const bool dot = dots && V.F.depth >= nu + 1;
    auto post = held ? k_amg_fuse_post<true> : k_amg_fuse_post<false>;
    post<<<V.fuse_blocks, AMG_FUSE_BLOCK, lds, ctx->stream>>>(
        F, nu, b, V.t, C.agg, C.e1, C.e2, C.kstep ? C.sc : nullptr, C.kstep ? C.part : nullptr, cnd, x,
        AMG_BJ_OMEGA, dot ? dots->a : nullptr, dot && dots->c_rhs ? 1 : 0, dot ? dots->y : nullptr,
        dot ? dots->part : nullptr);
    if (dot) dots->done = true;
    return;
  }
  float2 *cur = V.t, *oth = x;
  k_amg_bj<<<nb, BLOCK, 0, ctx->stream>>>(A, b, nullptr, cur, AMG_BJ_OMEGA);
  for (int s = 1; s < nu; s++) {
    k_amg_bj<<<nb, BLOCK, 0, ctx->stream>>>(A, b, cur, oth, AMG_BJ_OMEGA);
    std::swap(cur, oth);
  }
  AmgLevel &C = ctx->amg[l + 1];
  k_amg_residual<<<nb, BLOCK, 0, ctx->stream>>>(A, cur, b, V.r);
  k_amg_gather<<<nblk(C.n), BLOCK, 0, ctx->stream>>>(C.n, C.mptr, C.mem, V.r, nullptr, C.b);
  amg_solve_level(ctx, l + 1);
  k_amg_prolong<<<nb, BLOCK, 0, ctx->stream>>>(V.n, C.agg, C.e1, C.e2, AmgStep2{C.kstep ? C.sc : nullptr, nullptr, 0},
                                               cur, nullptr);
  for (int s = 0; s < nu; s++) {
    k_amg_bj<<<nb, BLOCK, 0, ctx->stream>>>(A, b, cur, oth, AMG_BJ_OMEGA);
    std::swap(cur, oth);
  }
}

// Levels l0..L-1 (no K-steps) as one V-cycle in one workgroup: A_l0 e1 = b
static void amg_tail_launch(ufe_ctx *ctx, int l0) {
  const int L = (int)ctx->amg.size();
  AmgTail T{};
  T.nlev = L - l0;
  int off = 0;
  for (int k = 0; k < T.nlev; k++) {
    AmgLevel &V = ctx->amg[l0 + k];
    T.L[k].A = amg_op(ctx, V);
    T.L[k].nnz = (int)V.nnz;
    T.L[k].mptr = V.mptr;
    T.L[k].mem = V.mem;
    T.L[k].agg = V.agg;
    T.L[k].nmem = V.nmem;
    T.L[k].lds = off;
    off += 3 * V.n;
  }
  // the two images follow the vectors when the set-up made room for them
  size_t bytes = ((size_t)off * sizeof(float2) + 15) & ~(size_t)15;
  T.imgA = T.imgB = nullptr;
  if (ctx->amg_tail_imgA) {
    T.imgA = ctx->amg_T ? ctx->amg_tail_imgAT : ctx->amg_tail_imgA;
    T.imgB = ctx->amg_tail_imgB;
    T.wordsA = ctx->amg_tail_wA;
    T.wordsB = ctx->amg_tail_wB;
    T.ldsA = (int)bytes;
    T.ldsB = (int)(bytes + 16 * (size_t)ctx->amg_tail_wA);
    bytes += 16 * ((size_t)ctx->amg_tail_wA + ctx->amg_tail_wB);
    for (int k = 0; k < T.nlev; k++) {
      T.L[k].offA = ctx->amg_tail_offA[k];
      T.L[k].offB = ctx->amg_tail_offB[k];
    }
  }
  T.inv = ctx->amg_direct ? ctx->amg_inv : nullptr;
  T.trans = ctx->amg_T ? 1 : 0;
  T.coarse_sweeps = AMG_COARSE_SWEEPS;
  T.nu = std::max(1, ctx->amg_nu);
  T.omega = AMG_BJ_OMEGA;
  T.b_in = ctx->amg[l0].b;
  T.x_out = ctx->amg[l0].e1;
  if (T.imgA)
    k_amg_tail<true><<<1, AMG_TAIL_THREADS, bytes, ctx->stream>>>(T);
  else
    k_amg_tail<false><<<1, AMG_TAIL_THREADS, bytes, ctx->stream>>>(T);
}

// A_l e = b_l: one cycle into e1, or (kstep) two cycles combined by GCR(2),
// the coefficients left in sc[6], sc[7] for the prolongation
static void amg_solve_level(ufe_ctx *ctx, int l) {
  if (ctx->amg_tail_l0 > 0 && l == ctx->amg_tail_l0) {
    amg_tail_launch(ctx, l);
    return;
  }
  AmgLevel &V = ctx->amg[l];
  AmgDots d1{nullptr, false, V.w1, V.part, false};
  amg_cycle(ctx, l, V.b, V.e1, V.kstep ? &d1 : nullptr);
  if (!V.kstep) return;
  const AmgOp A = amg_op(ctx, V);
  const int nd = amg_dot_count(V);
  if (!d1.done) {
    if (V.blocks)
      k_amg_dot_blocks<<<V.fuse_blocks, AMG_FUSE_BLOCK, 0, ctx->stream>>>(A, V.F, V.e1, V.w1, V.b, nullptr, V.part);
    else
      k_amg_matvec_dot<<<nd, 256, 0, ctx->stream>>>(A, V.e1, V.w1, V.b, nullptr, V.part);
  }
  const bool fold = amg_fused_cycle(ctx, l) && nd <= ctx->amg_kfold_max;
  const AmgFold F2{V.w1, nd, V.part, V.sc, V.rc2};
  if (fold) {
    // the second cycle's pre-smoothing kernel finishes step 1
  } else if (l >= 2) {   // the step-1 sums in every block of the update (no launch of their own)
    k_amg_kfin1_axpy<<<nblk(V.n, 256), 256, 0, ctx->stream>>>(nd, V.part, V.sc, V.n, V.b, V.w1, V.rc2);
  } else {
    k_amg_kfin<<<1, 256, 0, ctx->stream>>>(nd, V.part, V.sc, 1);
    k_amg_axpy<<<nblk(V.n), BLOCK, 0, ctx->stream>>>(V.n, V.b, V.w1, V.sc, V.rc2);
  }
  AmgDots d2{V.w1, true, V.w2, V.part, false};
  if (fold)
    amg_cycle(ctx, l, V.b, V.e2, &d2, &F2);
  else
    amg_cycle(ctx, l, V.rc2, V.e2, &d2);
  if (!d2.done) {
    if (V.blocks)
      k_amg_dot_blocks<<<V.fuse_blocks, AMG_FUSE_BLOCK, 0, ctx->stream>>>(A, V.F, V.e2, V.w2, V.w1, V.rc2, V.part);
    else
      k_amg_matvec_dot<<<nd, 256, 0, ctx->stream>>>(A, V.e2, V.w2, V.w1, V.rc2, V.part);
  }
  // the step-2 coefficients: computed by the fused post-smoothing of the level
  // above from these partials, or here for the other prolongations
  if (!amg_fused_cycle(ctx, l - 1) && !(l == 1 && amg_late_kfin(ctx))) k_amg_kfin<<<1, 256, 0, ctx->stream>>>(nd, V.part, V.sc, 2);
}

// The coarse levels of one application (level 1's b in, e1, e2 and sc out)
// only touch fixed buffers, so they are captured once per mesh and smoothing
// count and replayed: about 170 small kernels become one graph launch.
static int amg_capture(ufe_ctx *ctx) {
  hipGraphExec_t &G = ctx->amg_T ? ctx->amg_graph_T : ctx->amg_graph;
  int &Gnu = ctx->amg_T ? ctx->amg_graph_T_nu : ctx->amg_graph_nu;
  if (G && Gnu == ctx->amg_nu) return UFE_OK;
  if (G) (void)hipGraphExecDestroy(G);
  G = nullptr;
  hipGraph_t g = nullptr;
  HIPCHK(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
  amg_solve_level(ctx, 1);
  const hipError_t e1 = hipGetLastError();
  const hipError_t e2 = hipStreamEndCapture(ctx->stream, &g);
  if (e1 != hipSuccess || e2 != hipSuccess) {
    ctx->err = std::string("multigrid graph capture: ") + hipGetErrorString(e1 != hipSuccess ? e1 : e2);
    if (g) (void)hipGraphDestroy(g);
    return UFE_HIP_ERROR;
  }
  hipGraphExec_t ex = nullptr;
  const hipError_t e3 = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e3 != hipSuccess) {
    ctx->err = std::string("multigrid graph instantiate: ") + hipGetErrorString(e3);
    return UFE_HIP_ERROR;
  }
  G = ex;
  Gnu = ctx->amg_nu;
  return UFE_OK;
}

// ---------------------------------------------------------------------------
// Patches (patch_host.h): whole sweeps in one launch
// ---------------------------------------------------------------------------
// Own points of a patch and threads of its workgroup.  A thread holds one row
// of each colour, so the largest colour of the computed rows must fit the
// workgroup (a patch set that does not fit is built again with 3/4 of the own
// points).  Larger patches recompute fewer halo rows (1.9 rows per own row at
// 736, 2.7 at 240); smaller ones fill the 256 CUs on a small mesh.  Measured,
// own points : threads, on the 1M linear solve / the 182k-vertex batch / the 50k
// Picard loop / a 30k one (ms; per-colour kernels 67.2 / 56.0 / 71.7 / 24.8):
// 240:256 69.7 / 52.6 / 59.9 / 19.2, 480:512 64.4 / 51.7 / 55.9 / 19.6, 640:512
// 60.0 / 49.1 / 55.7 / 19.7, 800:512 57.3 / 48.0 / 54.8 / 19.5, 1000:1024
// 63.7 / 49.3 / 54.8 / 19.7, 1900:1024 58.0 / 46.9 / 57.1 / 20.1.  736 instead of
// 800 leaves room for denser colours before the rebuild.
constexpr size_t PATCH_LDS_MAX = 64 * 1024;
constexpr size_t SOR_LDS_MAX = 156 * 1024;   // of the 160 KiB of a CU
constexpr int SOR_THREADS_MAX = 1024;        // of a workgroup of the SOR loop, one row of a colour each
constexpr int SOR_PATCH_MIN = 64;            // own points of a workgroup of the SOR loop, at least
constexpr int PATCH_CUS = 256;               // CUs of an MI355X
constexpr int PATCH_LARGE = 1 << 17;         // points from which the large patches fill the chip
// LDS of a smoothing: values, coefficients and columns of the slots beyond the sixth
static size_t patch_lds_bytes(int list, int ov) {
  return (size_t)list * sizeof(float2) + (size_t)ov * (sizeof(float2) + sizeof(uint16_t));
}
struct PatchShape {
  int own, bs;
};
static PatchShape patch_shape(const ufe_ctx *ctx, PatchKind k) {
  if (k == PATCH_SOR64) {            // at most one workgroup per CU; its width follows from the rows
    const int own = std::max(SOR_PATCH_MIN, (ctx->nA + SOR_PATCHES - 1) / SOR_PATCHES);
    return {own, 0};
  }
  if (ctx->nA >= PATCH_LARGE) {
    const int one = (ctx->nA + PATCH_CUS - 1) / PATCH_CUS;   // a workgroup for each CU
    return {one <= 800 ? one : 736, 512};
  }
  return {std::max(64, std::min(240, ctx->nA / 256)), 256};
}

// Device memory for the patches.  They are one of two ways to the same results, so
// where there is no room p stays null and the colour launches run instead.
extern "C++" template <typename T>
static int patch_alloc(ufe_ctx *ctx, T *&p, size_t n) {
  void *q = nullptr;
  const hipError_t e = hipMalloc(&q, std::max(n, (size_t)1) * sizeof(T));
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    return UFE_OK;
  }
  HIPCHK(ctx, e);
  ctx->allocs.push_back(q);
  p = static_cast<T *>(q);
  return UFE_OK;
}

// One patch set as it goes to the device: its nine arrays, each of all parts, in one
// piece (a copy for each array of 16 parts took longer than the walk)
struct PatchImage {
  std::unique_ptr<char[]> host;
  size_t total = 0, first[9];        // bytes, and where each array starts
};
extern "C++" template <typename F>
static void patch_arrays(PatchDev &P, F f) {
  f(0, &PatchHost::d, P.d);
  f(1, &PatchHost::rows, P.rows);
  f(2, &PatchHost::nptr, P.nptr);
  f(3, &PatchHost::sbase, P.sbase);
  f(4, &PatchHost::lcol, P.lcol);
  f(5, &PatchHost::ov_e, P.ov_e);
  f(6, &PatchHost::ovf, P.ovf);
  f(7, &PatchHost::ov_c, P.ov_c);
  f(8, &PatchHost::ncol, P.ncol);
}
static void patch_pack(std::vector<PatchHost> &parts, int threads, PatchImage &I) {
  std::vector<size_t> first[9];      // of each array: the first byte of each part
  PatchDev P{};
  I.total = 0;
  patch_arrays(P, [&](int k, auto field, auto *&p) {
    first[k].assign(1, I.first[k] = I.total);
    for (const PatchHost &H : parts) first[k].push_back(first[k].back() + (H.*field).size() * sizeof(*p));
    I.total = (first[k].back() + 255) / 256 * 256;
  });
  I.host.reset(new char[I.total]);
  const int n = (int)parts.size();
  amg_parts(n, (int)std::min<size_t>(std::min(n, threads), 1 + (I.total >> 20)), [&](int, int t0, int t1) {
    for (int t = t0; t < t1; t++) {
      patch_arrays(P, [&](int k, auto field, auto *&) {
        const auto &v = parts[t].*field;
        if (!v.empty()) std::memcpy(I.host.get() + first[k][t], v.data(), first[k][t + 1] - first[k][t]);
      });
      parts[t] = PatchHost{};
    }
  });
}
static int patch_upload(ufe_ctx *ctx, const PatchImage &I, PatchSet &S) {   // S.P.d null: no room
  char *base = nullptr;
  if (const int r = patch_alloc(ctx, base, I.total)) return r;
  if (!base) return UFE_OK;
  HIPCHK(ctx, hipMemcpyAsync(base, I.host.get(), I.total, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));   // the image goes with the caller
  patch_arrays(S.P, [&](int k, auto, auto *&p) {
    p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(base + I.first[k]);
  });
  return UFE_OK;
}

// One set of patches on the host, smaller ones until they fit the workgroup (S.bs 0: none do)
static void patch_find(const ufe_ctx *ctx, const PatchMesh &m, const std::vector<int32_t> &order, PatchKind k, int nu,
                       int threads, std::vector<PatchHost> &parts, PatchSet &S) {
  PatchShape sh = patch_shape(ctx, k);
  const bool sor = k == PATCH_SOR64;
  bool fits = false;
  for (int tries = 0; tries < 6 && !fits; tries++, sh.own = sh.own * 3 / 4) {
    if (!patch_build(m, order, sh.own, nu, k == PATCH_POST32, true, !sor, parts, sor ? SOR_THREADS_MAX : INT32_MAX,
                     threads))
      break;
    int group = 0;
    S.P = PatchDev{};
    for (const PatchHost &H : parts) {
      group = std::max(group, H.max_group);
      S.P.np += (int)H.d.size();
      S.P.cap = std::max(S.P.cap, H.max_list);
      S.P.cap_ov = std::max(S.P.cap_ov, H.max_ov);
      S.P.cap_ncs = std::max(S.P.cap_ncs, H.max_ncs);
      S.P.cap_neu = std::max(S.P.cap_neu, H.max_neu);
      S.P.cap_ncol = std::max(S.P.cap_ncol, H.max_ncol);
    }
    if (sor) {                         // the number of workgroups is bounded: wide enough ones or none
      sh.bs = group <= 256 ? 256 : group <= 512 ? 512 : SOR_THREADS_MAX;
      S.lds = patch_sor_lds(S.P, sh.bs == SOR_THREADS_MAX);
      fits = S.lds <= SOR_LDS_MAX;
      break;
    }
    S.lds = patch_lds_bytes(S.P.cap, S.P.cap_ov);
    fits = group <= sh.bs && S.lds <= PATCH_LDS_MAX;
  }
  S.bs = fits ? sh.bs : 0;
  if (fits && sor) patch_mark_shared(ctx->nA, parts);
}

// Builds the wanted patch sets that are not there yet: start() walks them on host
// threads of its own, side by side, and finish() takes them to the device, so that a
// multigrid set-up runs meanwhile.  The lists and the context's mesh outlive it.
static bool sor_patch_resident(ufe_ctx *ctx, const PatchSet &S);
class PatchWalk {
 public:
  PatchWalk(ufe_ctx *c, HostLists &l) : ctx(c), L(l) {}
  ~PatchWalk() { join(); }
  int start(std::initializer_list<PatchKind> kinds, int sweeps) {
    nu = sweeps;
    for (PatchKind k : kinds)
      if (!ctx->patch[k][nu - 1].built) todo.push_back(k);
    if (todo.empty()) return UFE_OK;
    if (const int r = host_lists(ctx, L)) return r;
    set.resize(todo.size());
    image.resize(todo.size());
    try {
      th = std::thread([this] { walk(); });
    } catch (const std::exception &) {
      walk();
    }
    return UFE_OK;
  }
  int finish() {
    join();
    if (todo.empty()) return UFE_OK;
    int r;
    if (!ctx->d_place && !place.empty()) {
      int32_t *d = nullptr;
      if ((r = patch_alloc(ctx, d, place.size()))) return r;
      if (d) HIPCHK(ctx, hipMemcpy(d, place.data(), sizeof(int32_t) * place.size(), hipMemcpyHostToDevice));
      ctx->cor_apart = apart;
      ctx->d_place = d;
    }
    for (size_t i = 0; i < todo.size(); i++) {
      PatchSet &S = set[i];
      ctx->paths.patch_sets++;
      if (S.bs) {
        if ((r = patch_upload(ctx, image[i], S))) return r;
        S.ok = S.P.d && (todo[i] != PATCH_SOR64 || sor_patch_resident(ctx, S));
      }
      S.built = true;
      ctx->patch[todo[i]][nu - 1] = S;
    }
    return UFE_OK;
  }

 private:
  ufe_ctx *ctx;
  HostLists &L;
  int nu = 1;
  std::vector<PatchKind> todo;
  std::vector<PatchSet> set;         // bs 0: the mesh does not fit, or no host memory
  std::vector<PatchImage> image;
  std::vector<int32_t> place;
  bool apart = false;
  std::thread th;
  void join() {
    if (th.joinable()) th.join();
  }
  void walk() noexcept {
    try {
      const int nA = ctx->nA, nk = (int)todo.size(), threads = patch_threads(nA), each = std::max(1, threads / nk);
      const PatchMesh m{nA, ctx->colour_start, ctx->colour_active, L.cptr.data(), L.deg.data(), L.col.data(), ctx->n_neu,
                        ctx->n_cor, L.nrow.data(), L.nptr.data(), L.ncol.data(), L.crow.data(), L.cptr2.data(),
                        L.ccol.data(), ctx->h_key.data(), ctx->h_mid.empty() ? nullptr : ctx->h_mid.data()};
      const std::vector<int32_t> order = patch_order(m);
      amg_parts(nk, std::min(nk, threads), [&](int, int i0, int i1) {
        for (int i = i0; i < i1; i++) try {
            std::vector<PatchHost> parts;
            patch_find(ctx, m, order, todo[i], nu, each, parts, set[i]);
            if (set[i].bs) patch_pack(parts, each, image[i]);
          } catch (const std::bad_alloc &) {   // the colour launches do without
            set[i].bs = 0;
          }
      });
      std::vector<int32_t> at(nA, 0), met(L.crow);
      for (int i = 0; i < ctx->n_neu; i++) at[L.nrow[i]] = i + 1;
      for (int i = 0; i < ctx->n_cor; i++) at[L.crow[i]] = -i - 1;
      met.insert(met.end(), L.ccol.begin(), L.ccol.end());
      std::sort(met.begin(), met.end());
      apart = std::adjacent_find(met.begin(), met.end()) == met.end();
      place = std::move(at);
    } catch (const std::exception &) {
      for (PatchSet &S : set) S.bs = 0;
    }
  }
};

// The smoothing of the multigrid cycle runs on patches (one or two sweeps; the
// per-colour kernels otherwise, or with UFE_AMG_PATCH=0 in the environment when
// the hierarchy is first used with this sweep count).
static int amg_patches_start(ufe_ctx *ctx, PatchWalk &walk) {
  const int nu = std::max(1, ctx->amg_nu);
  if (nu > 2) return UFE_OK;
  const char *off = std::getenv("UFE_AMG_PATCH");
  if (off && off[0] == '0') {
    for (PatchKind k : {PATCH_PRE32, PATCH_POST32}) ctx->patch[k][nu - 1].built = true;
    return UFE_OK;
  }
  return walk.start({PATCH_PRE32, PATCH_POST32}, nu);
}
// The hierarchy (ctx->amg_nu set) and, meanwhile, the patches of the fine smoothing
static int amg_prepare(ufe_ctx *ctx) {
  HostLists lists;
  PatchWalk walk(ctx, lists);
  int r;
  if ((r = amg_patches_start(ctx, walk)) || (r = amg_setup(ctx, lists)) || (r = walk.finish())) return r;
  const int nu = std::max(1, ctx->amg_nu);
  if (nu > 2 || !ctx->patch[PATCH_PRE32][nu - 1].ok || !ctx->patch[PATCH_POST32][nu - 1].ok) return UFE_OK;
  return patch_spaces([&](auto *&p) { return patch_alloc(ctx, p, (size_t)ctx->nA); }, ctx->amg_zt, ctx->amg_zu);
}
static bool amg_on_patches(const ufe_ctx *ctx) {
  const int nu = std::max(1, ctx->amg_nu);
  return nu <= 2 && ctx->patch[PATCH_PRE32][nu - 1].ok && ctx->patch[PATCH_POST32][nu - 1].ok && ctx->d_place &&
         ctx->amg_zt && ctx->amg_zu;
}

// One smoothing on patches: from zero with the fine residual into y (pre), or
// from zin with A z into y when y is given (post)
extern "C++" template <int BS, int WAVES, int NU>
static void patch_smooth_launch(ufe_ctx *ctx, bool post, float omega, const float2 *v, const float2 *zin, float2 *z,
                                float2 *y) {
  const PatchSet &S = ctx->patch[post ? PATCH_POST32 : PATCH_PRE32][NU - 1];
  const dim3 grid((S.P.np + 7) / 8 * 8), block(BS);
  const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
  // what the launch cannot do without, whatever the number of sweeps: per row the
  // coefficients with their 16-bit columns, the row's index and position, centre,
  // Sxy and right-hand side, z out, z in (post) and the residual or A z
  int64_t rows = 0;
  for (int c = 0; c < 5; c++) rows += ctx->colour_active[c];
  const double bytes = 10.0 * ctx->degsum + (double)rows * (36.0 + (post ? 8.0 : 0.0) + (y ? 8.0 : 0.0));
  rows *= NU;                        // the rate counts vertex-sweeps
  const float2 *cU = ctx->d_cU32, *EV = ctx->d_EV32;
  const float *Sxy = ctx->d_Sxy32;
  if (!post)
    timed_kernel_lds(ctx, bytes, rows, k_patch_smooth<float, BS, WAVES, NU, false, true, true, 1>, grid, block, S.lds, S.P, cU,
                     Sxy, EV, skip, omega, v, zin, z, y);
  else if (y)
    timed_kernel_lds(ctx, bytes, rows, k_patch_smooth<float, BS, WAVES, NU, true, false, true, 2>, grid, block, S.lds, S.P, cU,
                     Sxy, EV, skip, omega, v, zin, z, y);
  else
    timed_kernel_lds(ctx, bytes, rows, k_patch_smooth<float, BS, WAVES, NU, true, false, true, 0>, grid, block, S.lds, S.P, cU,
                     Sxy, EV, skip, omega, v, zin, z, y);
}
static void patch_smooth(ufe_ctx *ctx, bool post, float omega, const float2 *v, const float2 *zin, float2 *z,
                         float2 *y) {
  const int nu = std::max(1, ctx->amg_nu);
  const PatchSet &S = ctx->patch[post ? PATCH_POST32 : PATCH_PRE32][nu - 1];
  auto go = [&](auto one, auto two) {
    if (nu == 1) one(ctx, post, omega, v, zin, z, y);
    else two(ctx, post, omega, v, zin, z, y);
  };
  if (S.bs == 256) go(patch_smooth_launch<256, 2, 1>, patch_smooth_launch<256, 2, 2>);
  else if (S.P.np <= PATCH_CUS) go(patch_smooth_launch<512, 2, 1>, patch_smooth_launch<512, 2, 2>);
  else go(patch_smooth_launch<512, 4, 1>, patch_smooth_launch<512, 4, 2>);
}

// z ~ A^-1 v on the fine level: nu forward FP32 SOR sweeps from zero, the
// coarse correction of the fine residual, nu backward sweeps; z leaves with
// the Neumann condition on the edge rows, like the SOR preconditioner's.
// w given: A z as well, when the smoothing computes it (returns whether it did).
static bool amg_apply(ufe_ctx *ctx, const AaAcMesh &am, float omega, const float2 *v, float2 *z,
                      float2 *w = nullptr) {
  const int n = ctx->nA, nu = std::max(1, ctx->amg_nu);
  const bool patches = amg_on_patches(ctx);
  AmgLevel &C = ctx->amg[1];
  (patches ? ctx->paths.smooth_patch : ctx->paths.smooth_colour)++;
  if (patches) {
    patch_smooth(ctx, false, omega, v, nullptr, ctx->amg_zt, ctx->amg_y);
  } else {
    // the first sweep starts from z = 0 (its first colour pass sets all of z).
    // The Neumann rows are brought up to date after the last sweep of each
    // smoothing only: the residual and the output need them, the smoother's own
    // sweeps converge as well with them one sweep behind (same iteration counts)
    for (int k = 0; k < nu; k++) enqueue_sweep_fp32(ctx, am, omega, z, v, false, false, k == nu - 1, k == 0);
    k_matvec_residual<<<nblk(n), BLOCK, 0, ctx->stream>>>(am, ctx->d_cU32, ctx->d_Sxy32, ctx->d_EV32,
                                                         active_ranges(ctx), z, v, ctx->amg_y);
  }
  k_amg_gather<<<nblk(C.n), BLOCK, 0, ctx->stream>>>(C.n, C.mptr, C.mem, ctx->amg_y, nullptr, C.b);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  (void)hipStreamIsCapturing(ctx->stream, &cap);
  // eager launches when the stream is being captured (recorded into the
  // caller's graph) or the graph launch is refused (the same kernels; the
  // refusal is cleared so that the launch checks after the cycle pass)
  bool launched = false;
  if (ctx->amg_graph && cap == hipStreamCaptureStatusNone) {
    launched = hipGraphLaunch(ctx->amg_graph, ctx->stream) == hipSuccess;
    if (!launched) (void)hipGetLastError();
  }
  if (!launched) amg_solve_level(ctx, 1);
  const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
  if (patches) {
    k_amg_prolong_neumann<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, C.agg, C.e1, C.e2, amg_fine_step2(ctx),
                                                             ctx->amg_zt, skip, ctx->amg_zu, neu_list(ctx),
                                                             cor_list(ctx), ctx->d_place);
    patch_smooth(ctx, true, omega, v, ctx->amg_zu, z, w);
    return w != nullptr;
  }
  k_amg_prolong<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, C.agg, C.e1, C.e2, amg_fine_step2(ctx), z, skip);
  neumann_f32(ctx, z);
  for (int k = 0; k < nu; k++) enqueue_sweep_fp32(ctx, am, omega, z, v, true, false, k == nu - 1);
  return false;
}

// The same for an FP64 Krylov method: the cycle runs in FP32 on rounded copies
static void amg_apply_f64(ufe_ctx *ctx, const AaAcMesh &am, float omega, const double2 *v, double2 *z) {
  const int n = ctx->nA;
  k_to_f32_pair<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, v, ctx->amg_v32);
  amg_apply(ctx, am, omega, ctx->amg_v32, ctx->amg_z32);
  k_to_f64_pair<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, ctx->amg_z32, z);
}

static void apply_AT(ufe_ctx *ctx, const AaAcMesh &mT, const ActiveRanges &ar, const double2 *x, double2 *y,
                     bool keep_fixed = false);
static void fold_T(ufe_ctx *ctx, double2 *y);
static RevList rev_list(ufe_ctx *c);

// The transposed smoothings run on the patches of the FP32 smoothing: A^T has the
// same neighbour lists (its zero couplings to edge points read points that stay
// zero), and the rows of the Neumann halo are computed along with the others.
static size_t patch_lds_bytes64(const PatchDev &P) {
  return (size_t)P.cap * sizeof(double2) + (size_t)P.cap_ov * (sizeof(double2) + sizeof(uint16_t));
}
static bool amg_T_on_patches(const ufe_ctx *ctx) {
  if (!amg_on_patches(ctx) || !ctx->amg_zt64) return false;
  const int nu = std::max(1, ctx->amg_nu);
  return patch_lds_bytes64(ctx->patch[PATCH_PRE32][nu - 1].P) <= PATCH_LDS_MAX &&
         patch_lds_bytes64(ctx->patch[PATCH_POST32][nu - 1].P) <= PATCH_LDS_MAX;
}
extern "C++" template <int BS, int NU>
static void patch_smooth_T_launch(ufe_ctx *ctx, const AaAcMesh &mT, bool post, double omega, const double2 *v,
                                  const double2 *zin, double2 *z, double2 *y) {
  const PatchSet &S = ctx->patch[post ? PATCH_POST32 : PATCH_PRE32][NU - 1];
  const dim3 grid((S.P.np + 7) / 8 * 8), block(BS);
  const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
  const size_t lds = patch_lds_bytes64(S.P);
  if (!post)
    k_patch_smooth<double, BS, 2, NU, false, true, false, 2><<<grid, block, lds, ctx->stream>>>(
        S.P, mT.cU, mT.Sxy, ctx->d_pair[1], skip, omega, v, zin, z, y);
  else
    k_patch_smooth<double, BS, 2, NU, true, false, false, 2><<<grid, block, lds, ctx->stream>>>(
        S.P, mT.cU, mT.Sxy, ctx->d_pair[1], skip, omega, v, zin, z, y);
}
// nu transposed sweeps from zero (forward) or from zin (post, backward) into z,
// and y = P^T A^T R^T z
static void patch_smooth_T(ufe_ctx *ctx, const AaAcMesh &mT, bool post, double omega, const double2 *v,
                           const double2 *zin, double2 *z, double2 *y) {
  const int nu = std::max(1, ctx->amg_nu);
  const bool narrow = ctx->patch[post ? PATCH_POST32 : PATCH_PRE32][nu - 1].bs == 256;
  auto go = narrow ? (nu == 1 ? patch_smooth_T_launch<256, 1> : patch_smooth_T_launch<256, 2>)
                   : (nu == 1 ? patch_smooth_T_launch<512, 1> : patch_smooth_T_launch<512, 2>);
  go(ctx, mT, post, omega, v, zin, z, y);
  const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
  const NeumannList E = neu_list(ctx), K = cor_list(ctx);
  if (E.n + K.n <= ctx->fold_max) {
    k_fold_T<<<1, FOLD_THREADS, 0, ctx->stream>>>(mT, E, K, rev_list(ctx), skip, z, y, ctx->cor_apart ? 1 : 0);
    return;
  }
  k_edge_rows_T<<<nblk(E.n + K.n), BLOCK, 0, ctx->stream>>>(mT, E, K, z, y);
  fold_T(ctx, y);
  if (skip) k_zero_skip_rows<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->nA, skip, y);
}

// The transposed operator P^T A^T R^T of the adjoint solves: nu forward FP64
// transposed SOR sweeps from zero (edge rows stay zero), the coarse correction
// on the transposed hierarchy (ctx->amg_T set by the caller), nu backward
// sweeps, and w = P^T A^T R^T z.
// On patches a smoothing with its operator product is 2 launches and reads the
// coefficients once; on colours it is 14 (40k vertices: 161 -> 66 us).
static void amg_apply_T(ufe_ctx *ctx, const AaAcMesh &mT, double omega, const double2 *v, double2 *z, double2 *w) {
  const int n = ctx->nA, nu = std::max(1, ctx->amg_nu);
  const bool patches = amg_T_on_patches(ctx);
  const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
  double2 *zt = patches ? ctx->amg_zt64 : z;   // between the smoothings
  auto sweep = [&](bool backward) {
    for (int i = 0; i < 5; i++) {
      const int c = backward ? 4 - i : i;
      const int m = ctx->colour_active[c];
      if (m == 0) continue;
      k_sor_colour<<<xcd_grid(m), BLOCK, 0, ctx->stream>>>(mT, z, ctx->d_pair[1], v, ctx->colour_start[c], m,
                                                         omega, nullptr, skip);
    }
  };
  AmgLevel &C = ctx->amg[1];
  (patches ? ctx->paths.smooth_T_patch : ctx->paths.smooth_T_colour)++;
  if (patches) {
    patch_smooth_T(ctx, mT, false, omega, v, nullptr, zt, ctx->amg_y64);
  } else {
    k_fill<double2><<<nblk(n), BLOCK, 0, ctx->stream>>>(z, n, make_double2(0.0, 0.0));
    for (int k = 0; k < nu; k++) sweep(false);
    apply_AT(ctx, mT, active_ranges(ctx), z, ctx->amg_y64);
  }
  k_amg_gather64<<<nblk(C.n), BLOCK, 0, ctx->stream>>>(C.n, C.mptr, C.mem, v, ctx->amg_y64, C.b);
  bool launched = false;
  if (ctx->amg_graph_T) {
    launched = hipGraphLaunch(ctx->amg_graph_T, ctx->stream) == hipSuccess;
    if (!launched) (void)hipGetLastError();
  }
  if (!launched) amg_solve_level(ctx, 1);   // the same kernels, eager
  k_amg_prolong64<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, C.agg, C.e1, C.e2, amg_fine_step2(ctx), zt, skip);
  if (patches) {
    patch_smooth_T(ctx, mT, true, omega, v, zt, z, w);
    return;
  }
  for (int k = 0; k < nu; k++) sweep(true);
  apply_AT(ctx, mT, active_ranges(ctx), z, w);
}

// colour passes of one multigrid application (for the sweep count)
static int64_t amg_passes(const ufe_ctx *ctx) { return 10 * (int64_t)std::max(1, ctx->amg_nu); }

// solve_SSA_linearised sweep loop (:601-691): returns the flags at exit.
// nb reference FP64 sweeps.  When the library is not sampling kernel times, a
// batch of 2^k sweeps (k < 8) is captured once as a HIP graph (the sweeps'
// kernels and their arguments: omega, tolerance, sweep limit, skip mask) and
// replayed with one launch; on small meshes the per-kernel launch costs more
// than the sweep's work.  The kernels are the same, so are the results.
// UFE_SOR_GRAPH=0 in the environment keeps eager launches.
static int sor_batch(ufe_ctx *ctx, const AaAcMesh &m, double omega, double tol, int max_sweeps, int nb) {
  const char *env = std::getenv("UFE_SOR_GRAPH");
  const bool graphs = !(env && env[0] == '0');
  int k = 0;
  while (k < 8 && (1 << k) < nb) k++;
  const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
  if (!graphs || ctx->prof || k >= 8 || (1 << k) != nb) {
    for (int b = 0; b < nb; b++) enqueue_sweep_fp64(ctx, m, omega, tol, max_sweeps);
    LAUNCHCHK(ctx);
    return UFE_OK;
  }
  ufe_ctx::SorGraph &G = ctx->sor_graph[k];
  if (!G.exec || G.omega != omega || G.tol != tol || G.max_sweeps != max_sweeps || G.skip != skip) {
    if (G.exec) (void)hipGraphExecDestroy(G.exec);
    G = ufe_ctx::SorGraph{};
    hipGraph_t g = nullptr;
    HIPCHK(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    for (int b = 0; b < nb; b++) enqueue_sweep_fp64(ctx, m, omega, tol, max_sweeps);
    const hipError_t e1 = hipGetLastError();
    const hipError_t e2 = hipStreamEndCapture(ctx->stream, &g);
    hipGraphExec_t ex = nullptr;
    const hipError_t e3 = (e1 == hipSuccess && e2 == hipSuccess) ? hipGraphInstantiate(&ex, g, nullptr, nullptr, 0)
                                                                 : hipErrorUnknown;
    if (g) (void)hipGraphDestroy(g);
    if (e1 != hipSuccess || e2 != hipSuccess || e3 != hipSuccess) {
      ctx->err = std::string("reference sweep graph: ") +
                 hipGetErrorString(e1 != hipSuccess ? e1 : (e2 != hipSuccess ? e2 : e3));
      return UFE_HIP_ERROR;
    }
    G.exec = ex;
    G.nb = nb;
    G.omega = omega;
    G.tol = tol;
    G.max_sweeps = max_sweeps;
    G.skip = skip;
  }
  HIPCHK(ctx, hipGraphLaunch(G.exec, ctx->stream));
  return UFE_OK;
}

// The buffers of the sweep loop on patches; sor_ready stays false where there is no room
static int sor_spaces(ufe_ctx *ctx) {
  auto vectors = [&](auto *&p) { return patch_alloc(ctx, p, (size_t)ctx->nA); };
  auto words = [&](auto *&p) { return patch_alloc(ctx, p, (size_t)SOR_REPORT_WORDS); };
  int r;
  if ((r = patch_spaces(vectors, ctx->sor_w1, ctx->sor_start)) || (r = patch_spaces(words, ctx->sor_reports))) return r;
  if (!ctx->sor_w1 || !ctx->sor_start || !ctx->sor_reports) return UFE_OK;
  k_fill<uint32_t><<<nblk(SOR_REPORT_WORDS), BLOCK, 0, ctx->stream>>>(ctx->sor_reports, SOR_REPORT_WORDS, 0u);
  LAUNCHCHK(ctx);
  ctx->sor_epoch = 0;
  ctx->sor_ready = true;
  return UFE_OK;
}

static const void *sor_patch_kernel(int bs) {
  return bs == 256 ? reinterpret_cast<const void *>(&k_patch_sor<256, false>)
         : bs == 512 ? reinterpret_cast<const void *>(&k_patch_sor<512, false>)
                     : reinterpret_cast<const void *>(&k_patch_sor<1024, true>);
}
// The errors by which the runtime declines a cooperative launch: the device has
// one cooperative queue, and a process beside one that holds it gets
// hipErrorIllegalState.  Nothing has run then, and the colour launches do the
// solve.  Any other error is an error of the call.
constexpr bool sor_launch_declined(hipError_t e) {
  return e == hipErrorIllegalState || e == hipErrorNotSupported || e == hipErrorCooperativeLaunchTooLarge;
}
static_assert(sor_launch_declined(hipErrorIllegalState) && !sor_launch_declined(hipSuccess) &&
                  !sor_launch_declined(hipErrorInvalidValue) && !sor_launch_declined(hipErrorOutOfMemory) &&
                  !sor_launch_declined(hipErrorLaunchFailure) && !sor_launch_declined(hipErrorIllegalAddress),
              "only what declines the launch itself may lead to the colour launches");
// Whether this process gets cooperative launches on the device, asked before any
// patch of the loop is built: where it does not, the building and the device
// memory would be for nothing.  Asked with a launch that has no patch, once per
// process and device, since the queue that decides it is the process's (a declined
// request takes 40 ms, the first accepted one 4).
static int sor_launch_offered(ufe_ctx *ctx, bool *yes) {
  static std::mutex lock;
  static std::map<int, bool> offered;
  const std::lock_guard<std::mutex> guard(lock);
  const auto known = offered.find(ctx->device);
  if (known != offered.end()) {
    *yes = known->second;
    return UFE_OK;
  }
  int coop = 0;
  HIPCHK(ctx, hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, ctx->device));
  hipError_t e = hipErrorNotSupported;
  if (coop) {
    PatchDev P{};
    const double2 *cU = nullptr;
    const double *Sxy = nullptr;
    const uint8_t *skip = nullptr;
    double x = 1.0;
    int n = 0;
    double2 *W = nullptr;
    uint32_t *reports = nullptr, epoch = 0;
    SorFlags *fl = nullptr;
    void *args[] = {&P, &cU, &Sxy, &cU, &cU, &skip, &x, &x, &n, &n, &n, &n, &W, &W, &W, &reports, &epoch, &fl};
    e = hipLaunchCooperativeKernel(sor_patch_kernel(256), dim3(8), dim3(256), args, 0, ctx->stream);
    if (sor_launch_declined(e)) (void)hipGetLastError();
    else HIPCHK(ctx, e);
  }
  offered[ctx->device] = *yes = e == hipSuccess;
  return UFE_OK;
}

// The sweep loop on patches (k_patch_sor): one launch per solve instead of seven
// per sweep, the same sweeps and bits.  Not used while kernel times are sampled
// (the sample is per colour launch), on meshes whose patches exceed a workgroup
// (about 230,000 vertices), where cooperative launches are declined, or with
// UFE_SOR_PATCH=0 in the environment when the mesh is first swept.  Returns the
// set, or null.
static const PatchSet *sor_patches(ufe_ctx *ctx, int *err) {
  *err = UFE_OK;
  if (ctx->prof) return nullptr;
  PatchSet &S = ctx->patch[PATCH_SOR64][0];
  if (!S.built) {
    const char *off = std::getenv("UFE_SOR_PATCH");
    if (off && off[0] == '0') {
      S.built = true;
      return nullptr;
    }
    const int own = patch_shape(ctx, PATCH_SOR64).own;
    if (patch_least_group(ctx->colour_active, (ctx->nA + own - 1) / own) > SOR_THREADS_MAX) {
      S.built = true;                // found from the colours, before anything is read back or walked
      return nullptr;
    }
    bool offered = false;
    if ((*err = sor_launch_offered(ctx, &offered))) return nullptr;
    if (!offered) {
      S.built = true;
      return nullptr;
    }
    HostLists lists;
    PatchWalk walk(ctx, lists);
    if ((*err = walk.start({PATCH_SOR64}, 1)) || (*err = walk.finish())) return nullptr;
  }
  if (S.ok && !ctx->sor_ready) {
    if ((*err = sor_spaces(ctx))) return nullptr;
    if (!ctx->sor_ready) S.ok = false;
  }
  return S.ok ? &S : nullptr;
}
// Whether the device keeps all workgroups of the loop resident
static bool sor_patch_resident(ufe_ctx *ctx, const PatchSet &S) {
  int cus = 0, per = 0;
  const void *k = sor_patch_kernel(S.bs);
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess ||
      // the limit belongs to the kernel and not to this mesh: never less than another mesh's patches need
      hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)SOR_LDS_MAX) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, S.bs, S.lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return S.P.np <= SOR_PATCHES && (S.P.np + 7) / 8 * 8 <= per * cus;
}

// Polls after which a workgroup of the loop gives up (about a second; a sweep's
// exchange takes a few).  UFE_SOR_SPINS=n in the environment sets it.
constexpr int SOR_SPINS = 1 << 20;
static int sor_spins() {
  const char *e = std::getenv("UFE_SOR_SPINS");
  char *end = nullptr;
  const long n = e ? std::strtol(e, &end, 10) : 0;
  return end == e || n < 0 ? SOR_SPINS : (int)std::min(n, 1l << 30);
}

static int run_sor_reference(ufe_ctx *ctx, double tol, int max_sweeps, SorFlags *out, double *seconds) {
  const AaAcMesh m = aaac_mesh(ctx);
  const double omega = ctx->params.SSA_SOR_omega;
  k_sor_flags_init<<<1, 1, 0, ctx->stream>>>(ctx->d_flags, 0);
  LAUNCHCHK(ctx);
  int batch = ctx->params.sweep_batch > 0 ? ctx->params.sweep_batch : 1;
  int queued = 0;
  auto t0 = std::chrono::steady_clock::now();
  int perr;
  if (const PatchSet *S = max_sweeps > 0 ? sor_patches(ctx, &perr) : (perr = UFE_OK, nullptr)) {
    // a launch holds the device for its sweeps, so a long solve takes several
    int limit = ctx->params.sweep_batch > 0 ? ctx->params.sweep_batch : 1024, swept = 0, top = max_sweeps;
    int spins = sor_spins();
    PatchDev P = S->P;
    const double2 *cU = ctx->d_cU, *EV = ctx->d_pair[1], *RHS = ctx->d_pair[2];
    const double *Sxy = ctx->d_Sxy;
    const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
    double om = omega, tl = tol;
    int nA = ctx->nA;
    double2 *W0 = ctx->d_pair[0], *W1 = ctx->sor_w1, *start = ctx->sor_start;
    uint32_t *reports = ctx->sor_reports;
    SorFlags *fl = ctx->d_flags;
    bool refused = false, gave_up = false;
    while (true) {
      uint32_t epoch = ctx->sor_epoch;
      void *args[] = {&P, &cU, &Sxy, &EV, &RHS, &skip, &om, &tl, &top, &limit, &spins, &nA, &W0, &W1,
                      &start, &reports, &epoch, &fl};
      const hipError_t launch = hipLaunchCooperativeKernel(sor_patch_kernel(S->bs), dim3((P.np + 7) / 8 * 8),
                                                           dim3(S->bs), args, (unsigned)S->lds, ctx->stream);
      refused = sor_launch_declined(launch);
      if (refused) {                 // the colour launches go on, for this mesh from here on
        (void)hipGetLastError();
        ctx->patch[PATCH_SOR64][0].ok = false;
        queued = swept;
        break;
      }
      HIPCHK(ctx, launch);
      ctx->paths.sor_patch++;
      HIPCHK(ctx, hipMemcpyAsync(ctx->h_flags, ctx->d_flags, sizeof(SorFlags), hipMemcpyDeviceToHost, ctx->stream));
      HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
      gave_up = ctx->h_flags->gave_up != 0;
      if (gave_up) {                 // from where this launch began, by colour launches; for this mesh from here on
        ctx->paths.sor_gave_up++;
        ctx->patch[PATCH_SOR64][0].ok = ctx->sor_ready = false;
        HIPCHK(ctx, hipMemcpyAsync(W0, start, sizeof(double2) * (size_t)nA, hipMemcpyDeviceToDevice, ctx->stream));
        k_sor_flags_init<<<1, 1, 0, ctx->stream>>>(ctx->d_flags, swept);
        LAUNCHCHK(ctx);
        queued = swept;
        break;
      }
      ctx->sor_epoch += (uint32_t)(ctx->h_flags->sweep - swept);
      swept = ctx->h_flags->sweep;
      if (ctx->h_flags->done || swept >= max_sweeps) break;
    }
    if (!refused && !gave_up) {
      if (seconds) *seconds += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
      *out = *ctx->h_flags;
      return UFE_OK;
    }
  } else if (perr) {
    return perr;
  }
  while (true) {
    const int nb = std::min(batch, max_sweeps - queued);
    int r;
    if ((r = sor_batch(ctx, m, omega, tol, max_sweeps, nb))) return r;
    ctx->paths.sor_colour++;
    queued += nb;
    HIPCHK(ctx, hipMemcpyAsync(ctx->h_flags, ctx->d_flags, sizeof(SorFlags), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    prof_collect(ctx);
    if (ctx->h_flags->done || queued >= max_sweeps) break;
    if (ctx->params.sweep_batch <= 0) batch = std::min(batch * 2, 64);
  }
  auto t1 = std::chrono::steady_clock::now();
  if (seconds) *seconds += std::chrono::duration<double>(t1 - t0).count();
  *out = *ctx->h_flags;
  return UFE_OK;
}

// ---- solve_SSA ---------------------------------------------------------------
static int ssa_viscosity_rn(ufe_ctx *ctx, double *RN) {
  const AaAcMesh m = aaac_mesh(ctx);
  SSAFields f = ssa_fields(ctx);
  const int nb = nblk(ctx->nA);
  k_ssa_viscosity<<<nb, BLOCK, 0, ctx->stream>>>(m, f, ctx->params.m_enh_ssa * 0.5, ctx->d_part);
  k_ssa_rn<<<1, 1024, 0, ctx->stream>>>(nb, ctx->d_part, ctx->d_scalar);
  LAUNCHCHK(ctx);
  if (RN) {
    HIPCHK(ctx, hipMemcpyAsync(ctx->h_scalar, ctx->d_scalar, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    *RN = ctx->h_scalar[0];
  }
  return UFE_OK;
}

static int ssa_prepare_coeffs(ufe_ctx *ctx) {
  k_ssa_prepare<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(aaac_mesh(ctx), ssa_fields(ctx), std::pow(100.0, 0.30));
  LAUNCHCHK(ctx);
  return UFE_OK;
}

static int ssa_gather(ufe_ctx *ctx) {
  k_ssa_gather<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(
      aaac_mesh(ctx), ssa_fields(ctx), F(ctx, "Hi"), F(ctx, "Hb"), F(ctx, "SL"), F(ctx, "dHs_dx_shelf"),
      F(ctx, "dHs_dy_shelf"), F(ctx, "A_flow_mean"), F(ctx, "U_SSA"), F(ctx, "V_SSA"), F(ctx, "Hi_Ac"),
      F(ctx, "Hb_Ac"), F(ctx, "SL_Ac"), F(ctx, "dHs_dx_shelf_Ac"), F(ctx, "dHs_dy_shelf_Ac"),
      F(ctx, "A_flow_mean_Ac"), F(ctx, "Ux_SSA_Ac"), F(ctx, "Uy_SSA_Ac"), ctx->params.use_tau_c_override);
  LAUNCHCHK(ctx);
  return UFE_OK;
}

static int ssa_finish(ufe_ctx *ctx) {
  k_ssa_finish<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(
      aaac_mesh(ctx), ac_mesh(ctx), ctx->d_pair[0], F(ctx, "U_SSA"), F(ctx, "V_SSA"), F(ctx, "Ux_SSA_Ac"),
      F(ctx, "Uy_SSA_Ac"), F(ctx, "Up_SSA_Ac"), F(ctx, "Uo_SSA_Ac"));
  LAUNCHCHK(ctx);
  return UFE_OK;
}

// calculate_GL_flux (:848-949): the grounding-line Ac velocities into W, the
// GL fluxes and the skip mask of the rows they prescribe
static int gl_prescribe(ufe_ctx *ctx) {
  GLFields g;
  g.Hi = F(ctx, "Hi"); g.Hb = F(ctx, "Hb"); g.SL = F(ctx, "SL"); g.Am = F(ctx, "A_flow_mean");
  g.sheet = FI(ctx, "mask_sheet"); g.phi = F(ctx, "phi_fric_AaAc"); g.iperm = ctx->d_iperm;
  g.glA = FI(ctx, "mask_gl_Ac");
  g.dHi_dx = F(ctx, "dHi_dx_Ac"); g.dHi_dy = F(ctx, "dHi_dy_Ac"); g.dSL_dx = F(ctx, "dSL_dx_Ac");
  g.dSL_dy = F(ctx, "dSL_dy_Ac"); g.dHb_dx = F(ctx, "dHb_dx_Ac"); g.dHb_dy = F(ctx, "dHb_dy_Ac");
  g.Qabs = F(ctx, "Qabs_GL_Ac"); g.Qp = F(ctx, "Qp_GL_Ac"); g.Ux = F(ctx, "Ux_SSA_Ac"); g.Uy = F(ctx, "Uy_SSA_Ac");
  g.W = ctx->d_pair[0];
  g.skip = ctx->d_skip;
  k_gl_flux<<<nblk(ctx->nAc), BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), g);
  LAUNCHCHK(ctx);
  return UFE_OK;
}

static int zero_ssa_outputs(ufe_ctx *ctx) {
  const char *aa[] = {"U_SSA", "V_SSA"};
  const char *ac[] = {"Ux_SSA_Ac", "Uy_SSA_Ac", "Up_SSA_Ac", "Uo_SSA_Ac"};
  for (auto n : aa) k_fill<double><<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(F(ctx, n), ctx->nV, 0.0);
  for (auto n : ac) k_fill<double><<<nblk(ctx->nAc), BLOCK, 0, ctx->stream>>>(F(ctx, n), ctx->nAc, 0.0);
  k_fill<double2><<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->d_pair[0], ctx->nA, make_double2(0.0, 0.0));
  LAUNCHCHK(ctx);
  return UFE_OK;
}

int ufe_solve_SSA(ufe_ctx *ctx, ufe_ssa_stats *st) try {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  ufe_ssa_stats local;
  if (!st) st = &local;
  std::memset(st, 0, sizeof(*st));
  const ufe_params &P = ctx->params;
  auto t0 = std::chrono::steady_clock::now();
  // gating (:430-465)
  HIPCHK(ctx, hipMemsetAsync(ctx->d_count, 0, sizeof(unsigned long long), ctx->stream));
  k_sum_int<<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(ctx->nV, FI(ctx, "mask_sheet"), ctx->d_count);
  LAUNCHCHK(ctx);
  unsigned long long nsheet = 0;
  HIPCHK(ctx, hipMemcpyAsync(ctx->h_scalar, ctx->d_count, sizeof(unsigned long long), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  std::memcpy(&nsheet, ctx->h_scalar, sizeof(nsheet));
  int r;
  if (P.ssa_forced_zero || nsheet == 0) {
    if ((r = zero_ssa_outputs(ctx))) return r;
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return UFE_OK;
  }
  if ((r = ssa_gather(ctx))) return r;
  // calculate_GL_flux (:471) prescribes the GL Ac velocities; SOR then skips
  // those rows (:627-631).  The Krylov solves treat them as fixed: their
  // residual and correction are zero, and every preconditioner leaves them
  // at zero, so the corrections never move the prescribed values.
  struct GLGuard {
    ufe_ctx *c;
    ~GLGuard() { c->gl_active = false; }
  } gl_guard{ctx};
  ctx->gl_active = P.use_analytical_GL_flux != 0;
  if (ctx->gl_active && (r = gl_prescribe(ctx))) return r;
  int it = 0, did_reset_before = 0, did_reset_now = 0;
  while (it < P.SSA_max_outer_loops) {
    it++;
    double RN = 0.0;
    if ((r = ssa_viscosity_rn(ctx, &RN))) return r;
    st->last_RN = RN;
    st->picard_iterations = it;
    if (RN < P.SSA_RN_tol) {
      st->picard_converged = 1;
      break;
    }
    if ((r = ssa_prepare_coeffs(ctx))) return r;
    if (P.precision != UFE_FP64) {
      // GMRES-IR to a relative residual, warm-started from the current velocities
      ufe_linsolve_opts lo{};
      lo.rel_tol = P.SSA_linear_rel_tol > 0.0 ? P.SSA_linear_rel_tol : 1e-6;
      lo.max_sweeps = 1 << 30;
      lo.precision = P.precision == UFE_MIXED ? UFE_MIXED : UFE_FP64;
      lo.gmres_restart = P.SSA_gmres_restart > 0 ? P.SSA_gmres_restart
                                                   : (P.SSA_precond_type == UFE_PRECOND_MULTIGRID ? 20 : 40);
      lo.precond_type = P.SSA_precond_type;
      lo.precond_sweeps = P.SSA_precond_sweeps > 0 ? P.SSA_precond_sweeps
                                                   : (P.SSA_precond_type == UFE_PRECOND_MULTIGRID ? 2 : 5);
      lo.orth_passes = 1;
      ufe_linsolve_stats ls;
      if ((r = ufe_ssa_linear_solve(ctx, &lo, &ls))) return r;
      if (it <= 64) st->sweeps[it - 1] = ls.sweeps;
      st->total_sweeps += ls.sweeps;
      st->last_max_residual = ls.rel_residual;
      st->sor_seconds += ls.seconds;
      if (ls.status != UFE_OK) st->status = UFE_SOR_NOT_CONVERGED;
      continue;
    }
    SorFlags fl;
    if ((r = run_sor_reference(ctx, P.SSA_max_residual_UV, P.SSA_max_inner_loops, &fl, &st->sor_seconds))) return r;
    if (it <= 64) st->sweeps[it - 1] = fl.sweep;
    st->total_sweeps += fl.sweep;
    st->last_max_residual = fl.last_maxres;
    if (fl.converged) did_reset_now = 0;
    if (fl.reset) {
      k_fill<double2><<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->d_pair[0], ctx->nA, make_double2(0.0, 0.0));
      LAUNCHCHK(ctx);
      did_reset_now = 1;
    }
    if (fl.hit_max && !fl.converged && !fl.reset) st->status = UFE_SOR_NOT_CONVERGED;
    if (did_reset_now) {
      st->resets++;
      if (!did_reset_before) did_reset_before = 1;
      else {
        ctx->err = "solve_SSA: SSA remains unstable after resetting velocities to zero";
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        return st->status = UFE_SSA_UNSTABLE;
      }
    }
  }
  if ((r = ssa_finish(ctx))) return r;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  st->total_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return st->status;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

// ---- linearised solve at fixed viscosity (bench path) ------------------------
int ufe_ssa_prepare(ufe_ctx *ctx) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  int r;
  if ((r = ssa_gather(ctx))) return r;
  if ((r = ssa_viscosity_rn(ctx, nullptr))) return r;
  if ((r = ssa_prepare_coeffs(ctx))) return r;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

// FP64 relative residual; with store=true also hands r to the FP32 sweeps.
// The FP64 relative residual with its block partial sums in `part` (at most
// sum over colours of nblk(rows) pairs) and the result in *scalar.
static int residual_fp64_into(ufe_ctx *ctx, double *part, double *scalar, double *rel, bool store) {
  const AaAcMesh m = aaac_mesh(ctx);
  const uint8_t *skip = ctx->gl_active ? ctx->d_skip : nullptr;
  int nb_tot = 0;
  for (int c = 0; c < 5; c++) {
    const int n = ctx->colour_active[c];
    if (!n) continue;
    const int nb = nblk(n);
    if (store)
      k_residual_store<<<nb, BLOCK, 0, ctx->stream>>>(m, ctx->d_pair[0], ctx->d_pair[1], ctx->d_pair[2],
                                                       ctx->colour_start[c], n, ctx->d_R32, part + 2 * nb_tot,
                                                       skip);
    else
      k_ssa_residual<<<nb, BLOCK, 0, ctx->stream>>>(m, ctx->d_pair[0], ctx->d_pair[1], ctx->d_pair[2],
                                                     ctx->colour_start[c], n, part + 2 * nb_tot, skip);
    nb_tot += nb;
  }
  k_ssa_rn<<<1, 1024, 0, ctx->stream>>>(nb_tot, part, scalar);
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipMemcpyAsync(ctx->h_scalar, scalar, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  *rel = ctx->h_scalar[0];
  return UFE_OK;
}

static int residual_fp64(ufe_ctx *ctx, double *rel, bool store = false) {
  const int r = residual_fp64_into(ctx, ctx->d_part, ctx->d_scalar, rel, store);
  if (r == UFE_OK) prof_collect(ctx);
  return r;
}

int ufe_ssa_residual(ufe_ctx *ctx, double *rel_residual) {
  if (!ctx || !ctx->have_mesh || !rel_residual) return UFE_BAD_INPUT;
  return residual_fp64(ctx, rel_residual);
}

static ActiveRanges active_ranges(ufe_ctx *ctx) {
  ActiveRanges a;
  for (int c = 0; c < 5; c++) {
    a.start[c] = ctx->colour_start[c];
    a.count[c] = ctx->colour_active[c];
  }
  a.skip = ctx->gl_active ? ctx->d_skip : nullptr;
  return a;
}

// The Krylov block read back to the host: H1 and H2 (65 x 64 each), Hs (65)
// and copies of d_scalar[0..2] (kry_g), in one device allocation, so that one
// copy into pinned memory brings all of it (four copies into pageable memory,
// each waiting for the one before, had left the device idle for about 0.1 ms
// per check).
constexpr size_t KRY_HBLOCK = 2 * 65 * 64 + 65 + 4;
static int kry_readback(ufe_ctx *ctx, const double **out) {
  if (!ctx->h_kry) {
    ctx->err = "the Krylov read-back buffer was not allocated";
    return UFE_HIP_ERROR;
  }
  k_copy_f64<<<1, 64, 0, ctx->stream>>>(3, ctx->d_scalar, ctx->kry_g);
  HIPCHK(ctx, hipMemcpyAsync(ctx->h_kry, ctx->kry_H1, sizeof(double) * KRY_HBLOCK, hipMemcpyDeviceToHost,
                             ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  *out = ctx->h_kry;
  return UFE_OK;
}

static int krylov_alloc(ufe_ctx *ctx, int m, bool f32) {
  if (ctx->kry_V && ctx->kry_m >= m && ctx->kry_f32 == f32) return UFE_OK;
  const size_t n = ctx->nA, es = f32 ? sizeof(float2) : sizeof(double2);
  int r;
  char *V, *Z, *w, *x;
  if ((r = dalloc(ctx, &V, es * n * (m + 1)))) return r;
  if ((r = dalloc(ctx, &Z, es * n * m))) return r;
  if ((r = dalloc(ctx, &w, es * n))) return r;
  if ((r = dalloc(ctx, &x, es * n))) return r;
  ctx->kry_V = V;
  ctx->kry_Z = Z;
  ctx->kry_w = w;
  ctx->kry_x = x;
  HIPCHK(ctx, hipMemsetAsync(V, 0, es * n * (m + 1), ctx->stream));
  if (!ctx->kry_R64 && (r = dalloc(ctx, &ctx->kry_R64, n))) return r;
  if (!ctx->kry_part && (r = dalloc(ctx, &ctx->kry_part, (size_t)64 * DOT_BLOCKS))) return r;
  if (!ctx->kry_H1) {   // one block, read back by one copy: H1, H2, Hs, the scalars
    if ((r = dalloc(ctx, &ctx->kry_H1, KRY_HBLOCK))) return r;
    ctx->kry_H2 = ctx->kry_H1 + 65 * 64;
    ctx->kry_Hs = ctx->kry_H2 + 65 * 64;
    ctx->kry_g = ctx->kry_Hs + 65;
    if ((r = dalloc(ctx, &ctx->kry_y, 65))) return r;
    if ((r = dalloc(ctx, &ctx->kry_nrm, 4))) return r;
  }
  // the block's pinned mirror, and 64 more for the least-squares solution
  // (kept with the context, across meshes)
  if (!ctx->h_kry) HIPCHK(ctx, hipHostMalloc((void **)&ctx->h_kry, sizeof(double) * (KRY_HBLOCK + 64)));
  ctx->kry_m = m;
  ctx->kry_f32 = f32;
  return UFE_OK;
}

// Least squares min |beta e1 - H y| for the (m+1) x m upper Hessenberg matrix
// of a GMRES cycle, by Givens rotations on the host.  Column j holds
// H(i,j) = H1[65 j + i] (+ H2[65 j + i]) for i <= j and H(j+1,j) = Hs[j].
// Returns the number of columns used (fewer on breakdown).
static int hessenberg_lsq(int m, const double *H1, const double *H2, const double *Hs, double beta,
                          std::vector<double> &y, double *resid = nullptr) {
  std::vector<double> H((size_t)(m + 1) * m, 0.0), g(m + 1, 0.0), cs(m), sn(m);
  auto Hat = [&](int i, int j) -> double & { return H[(size_t)j * (m + 1) + i]; };
  for (int j = 0; j < m; j++) {
    for (int i = 0; i <= j; i++) Hat(i, j) = H1[(size_t)j * 65 + i] + (H2 ? H2[(size_t)j * 65 + i] : 0.0);
    Hat(j + 1, j) = Hs[j];
  }
  g[0] = beta;
  int kk = m;
  for (int j = 0; j < m; j++) {
    for (int i = 0; i < j; i++) {
      const double a = cs[i] * Hat(i, j) + sn[i] * Hat(i + 1, j);
      const double b = -sn[i] * Hat(i, j) + cs[i] * Hat(i + 1, j);
      Hat(i, j) = a;
      Hat(i + 1, j) = b;
    }
    const double a = Hat(j, j), b = Hat(j + 1, j);
    const double rr = std::hypot(a, b);
    if (!(rr > 0.0) || !std::isfinite(rr)) { kk = j; break; }
    cs[j] = a / rr;
    sn[j] = b / rr;
    Hat(j, j) = rr;
    Hat(j + 1, j) = 0.0;
    g[j + 1] = -sn[j] * g[j];
    g[j] = cs[j] * g[j];
  }
  if (resid) *resid = std::fabs(g[kk]);
  y.assign(std::max(kk, 1), 0.0);
  for (int i = kk - 1; i >= 0; i--) {
    double t = g[i];
    for (int l = i + 1; l < kk; l++) t -= Hat(i, l) * y[l];
    y[i] = t / Hat(i, i);
  }
  return kk;
}

// colour passes of one preconditioner application of ks sweeps (the turn
// colour is skipped unless full sweeps were asked for)
static int64_t precond_passes(const ufe_ctx *ctx, int ks) {
  return 5 * (int64_t)ks - (ctx->repeat_turn ? 0 : (int64_t)(ks - 1));
}

// h = V^T w for k vectors
extern "C++" template <typename T>
static void orth_coeffs(ufe_ctx *ctx, int k, const ActiveRanges &ar, const typename V2T<T>::t *V,
                        const typename V2T<T>::t *w, double *h) {
  k_multi_dot<T><<<DOT_BLOCKS, BLOCK, 0, ctx->stream>>>(ctx->nA, k, ar, V, w, ctx->kry_part);
  k_multi_dot_reduce<<<k, 256, 0, ctx->stream>>>(DOT_BLOCKS, k, ctx->kry_part, h, 0);
}
// the last Gram-Schmidt pass: h = V^T w, w -= V h, next = w / |w| and the norm
extern "C++" template <typename T>
static void orth_step(ufe_ctx *ctx, int k, const ActiveRanges &ar, const typename V2T<T>::t *V,
                      typename V2T<T>::t *w, double *h, typename V2T<T>::t *next, double *norm) {
  orth_coeffs<T>(ctx, k, ar, V, w, h);
  k_multi_axpy_norm<T><<<DOT_BLOCKS, BLOCK, 0, ctx->stream>>>(ctx->nA, k, ar, V, h, w, ctx->kry_part);
  k_normalize_parts<T><<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->nA, w, DOT_BLOCKS, ctx->kry_part, next, norm);
}

// One GMRES(m) cycle on A d = r (r held in R32 or kry_R64 with |r|^2 in d_scalar[1]),
// then w += d in FP64.  Templated on the Krylov precision.  target > 0: every
// GMRES_CHECK iterations the least-squares residual is evaluated on the host
// and the cycle ends early once it has fallen below target |r|.
constexpr int GMRES_CHECK = 4;
extern "C++" template <typename T>
static int gmres_cycle(ufe_ctx *ctx, int m, int ksweeps, double omega, int passes, int64_t *cpass, int *matvecs,
                       double target = 0.0) {
  using T2 = typename V2T<T>::t;
  const bool f32 = sizeof(T) == 4;
  const int n = ctx->nA;
  const AaAcMesh am = aaac_mesh(ctx);
  const ActiveRanges ar = active_ranges(ctx);
  T2 *V = (T2 *)ctx->kry_V, *Z = (T2 *)ctx->kry_Z, *w = (T2 *)ctx->kry_w, *x = (T2 *)ctx->kry_x;
  const int nb = nblk(n);
  if (f32)
    k_r32_to_v<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_R32, ctx->d_scalar + 1, (float2 *)V);
  else
    k_r32_to_v64<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_R32, ctx->d_scalar + 1, (double2 *)V);
  if (!f32) {  // exact FP64 residual as v0 for the FP64 Krylov path
    k_residual_store64<<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_pair[0], ctx->d_pair[1], ctx->d_pair[2], ar,
                                                       ctx->kry_R64);
    k_normalize<double><<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->kry_R64, ctx->d_scalar + 1, (double2 *)V, ctx->kry_nrm + 1);
  }
  for (int j = 0; j < m; j++) {
    T2 *vj = V + (int64_t)j * n, *zj = Z + (int64_t)j * n;
    bool have_w = false;
    if (ctx->pc_amg) {
      if (f32) have_w = amg_apply(ctx, am, (float)omega, (const float2 *)vj, (float2 *)zj, (float2 *)w);
      else amg_apply_f64(ctx, am, (float)omega, (const double2 *)vj, (double2 *)zj);
      *cpass += amg_passes(ctx);
    } else {
      k_fill<T2><<<nb, BLOCK, 0, ctx->stream>>>(zj, n, T2{T(0), T(0)});
      for (int k = 0; k < ksweeps; k++) {
        const bool skip = k > 0 && !ctx->repeat_turn;
        const bool neu = !ctx->neumann_last || k == ksweeps - 1;
        if (f32) enqueue_sweep_fp32(ctx, am, (float)omega, (float2 *)zj, (const float2 *)vj, k & 1, skip, neu);
        else enqueue_sweep_fp64_vec(ctx, am, omega, (double2 *)zj, (const double2 *)vj, k & 1, skip, neu);
      }
      *cpass += precond_passes(ctx, ksweeps);
    }
    if (have_w) {
      // A z came with the post-smoothing
    } else if (f32)
      k_matvec<float><<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_cU32, ctx->d_Sxy32, ctx->d_EV32, ar, (const float2 *)zj, (float2 *)w);
    else
      k_matvec<double><<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_cU, ctx->d_Sxy, ctx->d_pair[1], ar, (const double2 *)zj, (double2 *)w);
    (*matvecs)++;
    // classical Gram-Schmidt, one or two passes
    double *h1 = ctx->kry_H1 + (int64_t)j * 65, *h2 = ctx->kry_H2 + (int64_t)j * 65;
    if (passes > 1) {
      orth_coeffs<T>(ctx, j + 1, ar, V, w, h1);
      k_multi_axpy<T><<<nb, BLOCK, 0, ctx->stream>>>(n, j + 1, V, h1, w);
    }
    orth_step<T>(ctx, j + 1, ar, V, w, passes > 1 ? h2 : h1, V + (int64_t)(j + 1) * n, ctx->kry_Hs + j);
    if (target > 0.0 && j + 1 < m && (j + 1) % GMRES_CHECK == 0) {
      const int k = j + 1;
      std::vector<double> yy;
      const double *hb = nullptr;
      if (const int e = kry_readback(ctx, &hb)) return e;
      double res = HUGE_VAL;
      const double beta = std::sqrt(hb[KRY_HBLOCK - 4 + 1]);
      hessenberg_lsq(k, hb, passes > 1 ? hb + 65 * 64 : nullptr, hb + 2 * 65 * 64, beta, yy, &res);
      if (res <= target * beta) {
        m = k;
        break;
      }
    }
  }
  LAUNCHCHK(ctx);
  // least squares min |beta e1 - H y| on the host (Givens rotations)
  const double *hb = nullptr;
  if (const int e = kry_readback(ctx, &hb)) return e;
  prof_collect(ctx);
  std::vector<double> y;
  const int kk = hessenberg_lsq(m, hb, passes > 1 ? hb + 65 * 64 : nullptr, hb + 2 * 65 * 64,
                                std::sqrt(hb[KRY_HBLOCK - 4 + 1]), y);
  if (kk == 0) return UFE_OK;
  double *hy = ctx->h_kry + KRY_HBLOCK;   // pinned: the copy reads it after this call returns
  std::copy(y.begin(), y.begin() + kk, hy);
  HIPCHK(ctx, hipMemcpyAsync(ctx->kry_y, hy, sizeof(double) * kk, hipMemcpyHostToDevice, ctx->stream));
  k_lincomb<T><<<nb, BLOCK, 0, ctx->stream>>>(n, kk, Z, ctx->kry_y, x);
  k_add_to_w<T><<<nb, BLOCK, 0, ctx->stream>>>(n, x, ctx->d_pair[0]);
  neumann_w(ctx);
  LAUNCHCHK(ctx);
  return UFE_OK;
}

// BiCGStab on A d = r (the FP64 residual, copied to precision T) until the
// recurrence residual falls by `reduce` or `max_sweeps` is reached; then
// w += d in FP64.  Vectors live in the Krylov work space, scalars in bic_S.
extern "C++" template <typename T>
static int bicg_inner(ufe_ctx *ctx, int ks, double omega, double reduce, int max_sweeps, int64_t *cpass,
                      int *matvecs) {
  using T2 = typename V2T<T>::t;
  const bool f32 = sizeof(T) == 4;
  const int n = ctx->nA, nb = nblk(n);
  const AaAcMesh am = aaac_mesh(ctx);
  const ActiveRanges ar = active_ranges(ctx);
  T2 *V = (T2 *)ctx->kry_V;
  T2 *rh = V, *r = V + (int64_t)n, *s = V + 2 * (int64_t)n, *t = V + 3 * (int64_t)n, *p = V + 4 * (int64_t)n,
     *v = V + 5 * (int64_t)n, *ph = V + 6 * (int64_t)n, *sh = V + 7 * (int64_t)n, *x = V + 8 * (int64_t)n;
  double *S = ctx->bic_S;
  if (f32) {
    k_bicg_init<float><<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_R32, (float2 *)rh, (float2 *)r, (float2 *)x,
                                                      (float2 *)p, (float2 *)v);
  } else {
    k_residual_store64<<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_pair[0], ctx->d_pair[1], ctx->d_pair[2], ar,
                                                       ctx->kry_R64);
    k_bicg_init<double><<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->kry_R64, (double2 *)rh, (double2 *)r,
                                                       (double2 *)x, (double2 *)p, (double2 *)v);
  }
  auto dot = [&](const T2 *a, int k, const T2 *b, double *out) {
    k_multi_dot<T><<<DOT_BLOCKS, BLOCK, 0, ctx->stream>>>(n, k, ar, a, b, ctx->kry_part);
    k_multi_dot_reduce<<<k, 256, 0, ctx->stream>>>(DOT_BLOCKS, k, ctx->kry_part, out, 0);
  };
  auto precond = [&](const T2 *in, T2 *out) {
    if (ctx->pc_amg) {
      if (f32) amg_apply(ctx, am, (float)omega, (const float2 *)in, (float2 *)out);
      else amg_apply_f64(ctx, am, (float)omega, (const double2 *)in, (double2 *)out);
      return;
    }
    k_fill<T2><<<nb, BLOCK, 0, ctx->stream>>>(out, n, T2{T(0), T(0)});
    for (int k = 0; k < ks; k++) {
      const bool skip = k > 0 && !ctx->repeat_turn;
      const bool neu = !ctx->neumann_last || k == ks - 1;
      if (f32) enqueue_sweep_fp32(ctx, am, (float)omega, (float2 *)out, (const float2 *)in, k & 1, skip, neu);
      else enqueue_sweep_fp64_vec(ctx, am, omega, (double2 *)out, (const double2 *)in, k & 1, skip, neu);
    }
  };
  auto matvec = [&](const T2 *in, T2 *out) {
    if (f32)
      k_matvec<float><<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_cU32, ctx->d_Sxy32, ctx->d_EV32, ar,
                                                     (const float2 *)in, (float2 *)out);
    else
      k_matvec<double><<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_cU, ctx->d_Sxy, ctx->d_pair[1], ar,
                                                      (const double2 *)in, (double2 *)out);
  };
  dot(rh, 2, r, S + 1);                       // rho = (r^, r), |r|^2
  k_bicg_scalars_init<<<1, 1, 0, ctx->stream>>>(S);
  LAUNCHCHK(ctx);
  double h[3];
  HIPCHK(ctx, hipMemcpyAsync(h, S + 1, 2 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  const double rr0 = h[1];
  if (!(rr0 > 0.0)) return UFE_OK;
  int it = 0;
  while (*cpass / 5 < max_sweeps) {
    k_bicg_beta<<<1, 1, 0, ctx->stream>>>(S);
    k_bicg_p<T><<<nb, BLOCK, 0, ctx->stream>>>(n, r, v, p, S);
    precond(p, ph);
    matvec(ph, v);
    dot(rh, 1, v, S + 5);
    k_bicg_alpha<<<1, 1, 0, ctx->stream>>>(S);
    k_bicg_s<T><<<nb, BLOCK, 0, ctx->stream>>>(n, r, v, s, S);
    precond(s, sh);
    matvec(sh, t);
    dot(s, 2, t, S + 6);                      // (s, t), (t, t): s and t are adjacent
    k_bicg_omega<<<1, 1, 0, ctx->stream>>>(S);
    k_bicg_update<T><<<nb, BLOCK, 0, ctx->stream>>>(n, ph, sh, s, t, x, r, S);
    dot(rh, 2, r, S + 1);                     // new rho and |r|^2: r^ and r are adjacent
    LAUNCHCHK(ctx);
    *cpass += 2 * (ctx->pc_amg ? amg_passes(ctx) : precond_passes(ctx, ks));
    *matvecs += 2;
    if (++it % 2 == 0) {
      HIPCHK(ctx, hipMemcpyAsync(h, S + 1, 2 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
      HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
      if (!std::isfinite(h[1]) || h[1] <= reduce * reduce * rr0) break;
    }
  }
  k_add_to_w<T><<<nb, BLOCK, 0, ctx->stream>>>(n, x, ctx->d_pair[0]);
  neumann_w(ctx);
  LAUNCHCHK(ctx);
  return UFE_OK;
}

int ufe_path_counts_get(ufe_ctx *ctx, ufe_path_counts *out) {
  if (!ctx || !out) return UFE_BAD_INPUT;
  *out = ctx->paths;
  return UFE_OK;
}

int ufe_multigrid_info_get(ufe_ctx *ctx, ufe_multigrid_info *out) {
  if (!ctx || !out) return UFE_BAD_INPUT;
  std::memset(out, 0, sizeof(*out));
  if (!ctx->amg_ready) return UFE_OK;
  const int L = std::min<int>((int)ctx->amg.size(), 16);
  out->levels = L;
  for (int l = 0; l < L; l++) {
    out->points[l] = ctx->amg[l].n;
    out->couplings[l] = ctx->amg[l].nnz;
    out->kstep[l] = ctx->amg[l].kstep ? 1 : 0;
    out->fused[l] = ctx->amg[l].fuse ? ctx->amg[l].F.depth : 0;
    out->fuse_list_max[l] = ctx->amg[l].fuse ? ctx->amg[l].F.cap : 0;
  }
  out->direct = ctx->amg_direct ? 1 : 0;
  out->setup_seconds = ctx->amg_setup_seconds;
  out->tail_level = ctx->amg_tail_l0;
  return UFE_OK;
}

int ufe_ssa_linear_solve(ufe_ctx *ctx, const ufe_linsolve_opts *o, ufe_linsolve_stats *st) try {
  if (!ctx || !ctx->have_mesh || !st || !o) return UFE_BAD_INPUT;
  std::memset(st, 0, sizeof(*st));
  const AaAcMesh m = aaac_mesh(ctx);
  const double omega = o->omega > 0.0 ? o->omega : ctx->params.SSA_SOR_omega;
  const int check = o->check_interval > 0 ? o->check_interval : 16;
  const bool mixed = o->precision == UFE_MIXED;
  ctx->repeat_turn = o->precond_full_sweeps != 0;
  ctx->neumann_last = o->precond_neumann_every_sweep == 0;
  auto t0 = std::chrono::steady_clock::now();
  double rel = 0.0;
  int r;
  const int mr = o->gmres_restart;
  if (mr < 0 || mr > 64) {
    ctx->err = "gmres_restart must be in 0..64";
    return UFE_BAD_INPUT;
  }
  if (o->precond_type != UFE_PRECOND_SOR && o->precond_type != UFE_PRECOND_MULTIGRID) {
    ctx->err = "precond_type must be UFE_PRECOND_SOR or UFE_PRECOND_MULTIGRID";
    return UFE_BAD_INPUT;
  }
  ctx->pc_amg = o->precond_type == UFE_PRECOND_MULTIGRID;
  if (ctx->pc_amg && o->method == 0 && mr == 0) {
    ctx->pc_amg = false;
    ctx->err = "the multigrid preconditioner needs a Krylov method (gmres_restart > 0 or BiCGStab)";
    return UFE_BAD_INPUT;
  }
  ctx->amg_nu = o->precond_sweeps > 0 ? o->precond_sweeps : 2;
  if (mixed || ctx->pc_amg) {  // FP32 centre coefficients of the current system (sweeps, FP32 cycle)
    k_to_f32_pair<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->nA, ctx->d_pair[1], ctx->d_EV32);
    LAUNCHCHK(ctx);
  }
  if (ctx->pc_amg) {
    ctx->amg_T = false;
    if ((r = amg_prepare(ctx))) return r;
    amg_refresh(ctx);
    LAUNCHCHK(ctx);
    if ((r = amg_capture(ctx))) return r;
  }
  if (o->method == 1) {
    // BiCGStab-IR: FP64 residual, inner BiCGStab in FP32 (mixed) or FP64
    if (ctx->n_neu) k_neumann_edges<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), ctx->d_pair[0], nullptr);
    k_neumann_scalar_pair_corners<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), ctx->d_pair[0]);
    const bool k32 = mixed;   // FP32 Krylov vectors
    if ((r = krylov_alloc(ctx, std::max(mr, 8), k32))) return r;
    if (!ctx->bic_S && (r = dalloc(ctx, &ctx->bic_S, 16))) return r;
    const int ks = o->precond_sweeps > 0 ? o->precond_sweeps : 2;
    if ((r = residual_fp64(ctx, &rel, mixed))) return r;
    st->refinements = 1;
    double prev = HUGE_VAL;
    int64_t cp = 0;
    while (rel > o->rel_tol && cp / 5 < o->max_sweeps) {
      if (rel > 0.99 * prev) break;
      prev = rel;
      const double reduce = std::max(0.1 * o->rel_tol / rel, k32 ? 1e-4 : 1e-13);
      r = k32 ? bicg_inner<float>(ctx, ks, omega, reduce, o->max_sweeps, &cp, &st->matvecs)
              : bicg_inner<double>(ctx, ks, omega, reduce, o->max_sweeps, &cp, &st->matvecs);
      st->sweeps = (int32_t)(cp / 5);
      if (r) return r;
      if ((r = residual_fp64(ctx, &rel, mixed))) return r;
      st->refinements++;
      if (!std::isfinite(rel)) break;
    }
    st->rel_residual = rel;
    st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    st->status = rel <= o->rel_tol ? UFE_OK : UFE_SOR_NOT_CONVERGED;
    return UFE_OK;
  }
  if (mr > 0) {
    // GMRES works on the Neumann-consistent subspace (edge rows follow the SOR
    // rows), which the corrections keep: start the velocities there as well
    if (ctx->n_neu) k_neumann_edges<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), ctx->d_pair[0], nullptr);
    k_neumann_scalar_pair_corners<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), ctx->d_pair[0]);
    const bool k32 = mixed;   // FP32 Krylov vectors
    if ((r = krylov_alloc(ctx, mr, k32))) return r;
    const int ks = o->precond_sweeps > 0 ? o->precond_sweeps : 2;
    if ((r = residual_fp64(ctx, &rel, true))) return r;
    st->refinements = 1;
    double prev = HUGE_VAL;
    int64_t cp = 0;
    while (rel > o->rel_tol && cp / 5 < o->max_sweeps) {
      if (rel > 0.99 * prev) break;   // stagnated at the rounding floor of the residual
      prev = rel;
      int mv = 0;
      const int passes = o->orth_passes > 0 ? o->orth_passes : 2;
      // end the cycle once its own residual estimate is half of what the tolerance asks
      const double target = 0.5 * o->rel_tol / rel;
      r = k32 ? gmres_cycle<float>(ctx, mr, ks, omega, passes, &cp, &mv, target)
              : gmres_cycle<double>(ctx, mr, ks, omega, passes, &cp, &mv, target);
      st->sweeps = (int32_t)(cp / 5);
      if (r) return r;
      st->matvecs += mv;
      if ((r = residual_fp64(ctx, &rel, true))) return r;
      st->refinements++;
      if (!std::isfinite(rel)) break;
    }
    st->rel_residual = rel;
    st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    st->status = rel <= o->rel_tol ? UFE_OK : UFE_SOR_NOT_CONVERGED;
    return UFE_OK;
  }
  if ((r = residual_fp64(ctx, &rel, mixed))) return r;
  st->refinements = 1;
  while (rel > o->rel_tol && st->sweeps < o->max_sweeps) {
    const int nb = std::min(check, o->max_sweeps - st->sweeps);
    if (mixed) {
      k_fill<float2><<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->d_D32, ctx->nA, make_float2(0.0f, 0.0f));
      for (int b = 0; b < nb; b++) enqueue_sweep_fp32(ctx, m, (float)omega);
      k_apply_correction<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->nA, ctx->d_D32, ctx->d_pair[0]);
      neumann_w(ctx);
    } else {
      for (int b = 0; b < nb; b++) enqueue_sweep_fp64(ctx, m, omega, 0.0, 1 << 30, false);
    }
    LAUNCHCHK(ctx);
    st->sweeps += nb;
    if ((r = residual_fp64(ctx, &rel, mixed))) return r;
    st->refinements++;
  }
  st->rel_residual = rel;
  st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  st->status = rel <= o->rel_tol ? UFE_OK : UFE_SOR_NOT_CONVERGED;
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}


// The plain FP64 SOR path of ufe_ssa_linear_solve with the residual's scratch
// in the file-scope array: the same kernels, launch shapes and summation
// order, so the same sweeps and bit-identical velocities.  Nothing is
// allocated: no hipMalloc, no events (kernel profiling is suspended for the
// call), the result is read through the context's pinned scalar.
int ufe_ssa_sor_solve_noalloc(ufe_ctx *ctx, double rel_tol, int32_t max_sweeps, double omega,
                              int32_t check_interval, ufe_linsolve_stats *st) try {
  if (!ctx || !ctx->have_mesh || !st) return UFE_BAD_INPUT;
  std::memset(st, 0, sizeof(*st));
  if (ctx->nA > NOALLOC_MAX_ROWS) {
    ctx->err = "ufe_ssa_sor_solve_noalloc: the mesh has more SOR rows (nVAaAc) than its scratch holds "
               "(at most 8388608)";
    return UFE_BAD_INPUT;
  }
  if (!ctx->noalloc_scratch) {
    ctx->err = "ufe_ssa_sor_solve_noalloc: no device address for the scratch array on this device";
    return UFE_HIP_ERROR;
  }
  double *part = ctx->noalloc_scratch, *scalar = ctx->noalloc_scratch + 2 * NOALLOC_PARTS;
  struct ProfPause {      // event pairs would be created on demand: none during this call
    ufe_ctx *c;
    bool was;
    ~ProfPause() { c->prof = was; }
  } pause{ctx, ctx->prof};
  ctx->prof = false;
  const AaAcMesh m = aaac_mesh(ctx);
  const double om = omega > 0.0 ? omega : ctx->params.SSA_SOR_omega;
  const int check = check_interval > 0 ? check_interval : 16;
  const auto t0 = std::chrono::steady_clock::now();
  double rel = 0.0;
  int r;
  if ((r = residual_fp64_into(ctx, part, scalar, &rel, false))) return r;
  st->refinements = 1;
  while (rel > rel_tol && st->sweeps < max_sweeps) {
    const int nb = std::min(check, max_sweeps - st->sweeps);
    for (int b = 0; b < nb; b++) enqueue_sweep_fp64(ctx, m, om, 0.0, 1 << 30, false);
    LAUNCHCHK(ctx);
    st->sweeps += nb;
    if ((r = residual_fp64_into(ctx, part, scalar, &rel, false))) return r;
    st->refinements++;
  }
  st->rel_residual = rel;
  st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  st->status = rel <= rel_tol ? UFE_OK : UFE_SOR_NOT_CONVERGED;
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

// ---- adjoint of the SSA solve ------------------------------------------------
// (no reference counterpart; the forward mirrors the Picard loop of
// src/ice_dynamics_module.f90:498-545 with tight linear solves)

static AaAcMesh aaac_mesh_T(ufe_ctx *ctx) {
  AaAcMesh m = aaac_mesh(ctx);
  m.cU = ctx->d_cUT;
  m.cNx = ctx->d_cNxT;
  m.cNy = ctx->d_cNyT;
  return m;
}
static RevList rev_list(ufe_ctx *c) {
  RevList R;
  R.n = c->n_rev;
  R.tgt = c->d_rev_tgt;
  R.ptr = c->d_rev_ptr;
  R.src = c->d_rev_src;
  R.cnt = c->d_rev_cnt;
  return R;
}

static int adj_alloc(ufe_ctx *ctx, int m, int K, int every) {
  const size_t n = ctx->nA;
  int r;
  if (!ctx->adj_V || ctx->adj_m < m) {
    if ((r = dalloc(ctx, &ctx->adj_V, n * (m + 1)))) return r;
    if ((r = dalloc(ctx, &ctx->adj_Z, n * m))) return r;
    ctx->adj_m = m;
  }
  if (!ctx->adj_w) {
    if ((r = dalloc(ctx, &ctx->adj_w, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_r, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_g, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_lam, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_ubar, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_uK, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_gs, 4 * n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_gtau, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_gA, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_pbar, n))) return r;
    if ((r = dalloc(ctx, &ctx->adj_H1, 65 * 64))) return r;
    if ((r = dalloc(ctx, &ctx->adj_Hs, 65))) return r;
    if ((r = dalloc(ctx, &ctx->adj_y, 65))) return r;
    if ((r = dalloc(ctx, &ctx->adj_nrm, 8))) return r;
    if (!ctx->kry_part && (r = dalloc(ctx, &ctx->kry_part, (size_t)64 * DOT_BLOCKS))) return r;
  }
  const int nck = (K + every - 1) / every;
  while ((int)ctx->adj_ck.size() < nck) {
    double2 *b;
    if ((r = dalloc(ctx, &b, n))) return r;
    ctx->adj_ck.push_back(b);
  }
  while ((int)ctx->adj_seg.size() < every - 1) {
    double2 *b;
    if ((r = dalloc(ctx, &b, n))) return r;
    ctx->adj_seg.push_back(b);
  }
  ctx->adj_nck = nck;
  return UFE_OK;
}

static int copy_pair(ufe_ctx *ctx, double2 *dst, const double2 *src) {
  HIPCHK(ctx, hipMemcpyAsync(dst, src, sizeof(double2) * ctx->nA, hipMemcpyDeviceToDevice, ctx->stream));
  return UFE_OK;
}

// one Picard step of the adjoint forward: eta, S and the system from W, then W := solution
static int adj_forward_step(ufe_ctx *ctx, int *sweeps, double *rel, int *status) {
  int r;
  if ((r = ssa_viscosity_rn(ctx, nullptr))) return r;
  if ((r = ssa_prepare_coeffs(ctx))) return r;
  ufe_linsolve_stats ls;
  if ((r = ufe_ssa_linear_solve(ctx, &ctx->adj_lin, &ls))) return r;
  *sweeps += ls.sweeps;
  *rel = std::max(*rel, ls.rel_residual);
  if (ls.status != UFE_OK) *status = ls.status;
  return UFE_OK;
}

// P^T: fold the edge rows of y back onto the SOR rows that define them, then clear them
static void fold_T(ufe_ctx *ctx, double2 *y) {
  k_fold_corners<<<1, 1, 0, ctx->stream>>>(cor_list(ctx), y);
  if (ctx->n_rev) k_fold_edges<<<nblk(ctx->n_rev), BLOCK, 0, ctx->stream>>>(rev_list(ctx), y);
  if (ctx->n_neu) k_zero_rows<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), y);
}
// y = P^T A^T R^T x.  With the grounding-line rows held fixed they are no
// unknowns of the system: `keep_fixed` false zeroes them in y, true keeps
// their values, which are the couplings of the prescribed velocities into the
// free rows' equations.
static void apply_AT(ufe_ctx *ctx, const AaAcMesh &mT, const ActiveRanges &ar, const double2 *x, double2 *y,
                     bool keep_fixed) {
  k_matvec_T<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(mT, ctx->d_pair[1], ar, x, y);
  fold_T(ctx, y);
  if (ctx->gl_active && !keep_fixed)
    k_zero_skip_rows<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->nA, ctx->d_skip, y);
}
// z = ks transposed SOR sweeps from zero on A^T z = v (edge rows stay zero)
static void precond_T(ufe_ctx *ctx, const AaAcMesh &mT, double omega, int ks, const double2 *v, double2 *z) {
  k_fill<double2><<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(z, ctx->nA, make_double2(0.0, 0.0));
  for (int k = 0; k < ks; k++)
    for (int i = k > 0 ? 1 : 0; i < 5; i++) {   // the turn colour once, as in the forward preconditioner
      const int c = (k & 1) ? 4 - i : i;
      const int n = ctx->colour_active[c];
      if (n == 0) continue;
      k_sor_colour<<<xcd_grid(n), BLOCK, 0, ctx->stream>>>(mT, z, ctx->d_pair[1], v, ctx->colour_start[c], n,
                                                         omega, nullptr, ctx->gl_active ? ctx->d_skip : nullptr);
    }
}

// restarted GMRES(m) on (P^T A^T R^T) lam = g, FP64, right-preconditioned by
// transposed SOR; lam (ctx->adj_lam) is the initial guess on entry
static int adj_solve(ufe_ctx *ctx, double tol, int m, int ks, double omega, int max_sweeps, int *sweeps,
                     int *matvecs, double *rel_out) {
  const int n = ctx->nA, nb = nblk(n);
  const AaAcMesh mT = aaac_mesh_T(ctx);
  const ActiveRanges ar = active_ranges(ctx);
  double2 *V = ctx->adj_V, *Z = ctx->adj_Z, *w = ctx->adj_w, *rr = ctx->adj_r;
  int used = 0;
  const bool mg = ctx->adj_lin.precond_type == UFE_PRECOND_MULTIGRID;
  if (mg) {                           // the transposed hierarchy for this system's diagonals
    int r;
    ctx->amg_T = false;
    ctx->amg_nu = ks;
    if ((r = amg_prepare(ctx))) return r;
    const char *fold = std::getenv("UFE_FOLD_MAX");
    ctx->fold_max = fold && *fold ? (int)std::strtol(fold, nullptr, 10) : FOLD_MAX;
    if (amg_on_patches(ctx) && !ctx->amg_zt64 && (r = patch_alloc(ctx, ctx->amg_zt64, (size_t)n))) return r;
    ctx->amg_T = true;
    k_to_f32_pair<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, ctx->d_pair[1], ctx->d_EV32);
    amg_refresh(ctx);
    LAUNCHCHK(ctx);
    r = amg_capture(ctx);
    if (r) {
      ctx->amg_T = false;
      return r;
    }
  }
  struct ResetT {                     // back to the forward orientation on every exit
    ufe_ctx *c;
    ~ResetT() { c->amg_T = false; }
  } reset_t{ctx};
  double rel = 0.0, prev = HUGE_VAL;
  std::vector<double> H1(65 * 64), Hs(65), sc(4);
  while (true) {
    apply_AT(ctx, mT, ar, ctx->adj_lam, w);
    k_adj_residual<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->adj_g, w, rr, ctx->d_part);
    k_adj_norms<<<1, 1024, 0, ctx->stream>>>(nb, ctx->d_part, ctx->adj_nrm);
    LAUNCHCHK(ctx);
    HIPCHK(ctx, hipMemcpyAsync(sc.data(), ctx->adj_nrm, sizeof(double) * 3, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    const double gn = std::sqrt(sc[2]);
    rel = gn > 0.0 ? sc[0] / gn : 0.0;
    if (!std::isfinite(rel)) {
      ctx->err = "adjoint solve diverged";
      return UFE_SOR_NOT_CONVERGED;
    }
    if (rel <= tol || gn == 0.0 || used >= max_sweeps) break;
    if (rel > 0.99 * prev) break;   // stagnated at the rounding floor of the residual
    prev = rel;
    k_normalize<double><<<nb, BLOCK, 0, ctx->stream>>>(n, rr, ctx->adj_nrm + 1, V, ctx->adj_nrm + 4);
    for (int j = 0; j < m; j++) {
      double2 *vj = V + (int64_t)j * n, *zj = Z + (int64_t)j * n;
      if (mg) {
        amg_apply_T(ctx, mT, omega, vj, zj, w);
      } else {
        precond_T(ctx, mT, omega, ks, vj, zj);
        apply_AT(ctx, mT, ar, zj, w);
      }
      used += mg ? 2 * ks : ks;
      (*matvecs)++;
      orth_step<double>(ctx, j + 1, ar, V, w, ctx->adj_H1 + (int64_t)j * 65, V + (int64_t)(j + 1) * n, ctx->adj_Hs + j);
    }
    LAUNCHCHK(ctx);
    HIPCHK(ctx, hipMemcpyAsync(H1.data(), ctx->adj_H1, sizeof(double) * 65 * m, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipMemcpyAsync(Hs.data(), ctx->adj_Hs, sizeof(double) * m, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    std::vector<double> y;
    const int kk = hessenberg_lsq(m, H1.data(), nullptr, Hs.data(), sc[0], y);
    if (kk == 0) break;
    HIPCHK(ctx, hipMemcpyAsync(ctx->adj_y, y.data(), sizeof(double) * kk, hipMemcpyHostToDevice, ctx->stream));
    k_lincomb<double><<<nb, BLOCK, 0, ctx->stream>>>(n, kk, Z, ctx->adj_y, w);
    k_add_pair<<<nb, BLOCK, 0, ctx->stream>>>(n, w, ctx->adj_lam);
    LAUNCHCHK(ctx);
  }
  *sweeps += used;
  *rel_out = rel;
  return rel <= tol ? UFE_OK : UFE_SOR_NOT_CONVERGED;
}

int ufe_ssa_adjoint_forward(ufe_ctx *ctx, const ufe_adjoint_opts *o, ufe_adjoint_stats *st) try {
  if (!ctx || !ctx->have_mesh || !o || !st) return UFE_BAD_INPUT;
  std::memset(st, 0, sizeof(*st));
  if (o->picard_iterations < 1 || o->picard_iterations > 100000 || o->checkpoint_every < 1 ||
      o->gmres_restart < 1 || o->gmres_restart > 64 || !(o->lin_rel_tol > 0.0) ||
      (o->precision != UFE_FP64 && o->precision != UFE_MIXED) ||
      (o->precond_type != UFE_PRECOND_SOR && o->precond_type != UFE_PRECOND_MULTIGRID)) {
    ctx->err = "ufe_ssa_adjoint_forward: picard_iterations >= 1, checkpoint_every >= 1, gmres_restart in 1..64, "
               "lin_rel_tol > 0 and precision UFE_FP64 or UFE_MIXED are required";
    return UFE_BAD_INPUT;
  }
  const int K = o->picard_iterations, every = o->checkpoint_every;
  int r;
  if ((r = adj_alloc(ctx, o->gmres_restart, K, every))) return r;
  ufe_linsolve_opts &L = ctx->adj_lin;
  L = ufe_linsolve_opts{};
  L.rel_tol = o->lin_rel_tol;
  L.max_sweeps = o->max_sweeps > 0 ? o->max_sweeps : 1000000;
  L.precision = o->precision;
  L.omega = o->omega;
  L.gmres_restart = o->gmres_restart;
  L.precond_sweeps = o->precond_sweeps;
  L.precond_type = o->precond_type;
  L.orth_passes = 1;
  ctx->adj_ready = false;
  auto t0 = std::chrono::steady_clock::now();
  if ((r = ssa_gather(ctx))) return r;
  // with the GL flux (:471) the grounding-line rows hold its velocities in
  // every Picard step, as in solve_SSA
  struct GLGuard {
    ufe_ctx *c;
    ~GLGuard() { c->gl_active = false; }
  } gl_guard{ctx};
  ctx->adj_gl = ctx->params.use_analytical_GL_flux != 0;
  ctx->gl_active = ctx->adj_gl;
  if (ctx->adj_gl && (r = gl_prescribe(ctx))) return r;
  for (int k = 1; k <= K; k++) {
    if ((k - 1) % every == 0) {
      if ((r = copy_pair(ctx, ctx->adj_ck[(k - 1) / every], ctx->d_pair[0]))) return r;
      st->checkpoints++;
    }
    if ((r = adj_forward_step(ctx, &st->forward_sweeps, &st->max_forward_residual, &st->status))) return r;
  }
  if ((r = copy_pair(ctx, ctx->adj_uK, ctx->d_pair[0]))) return r;
  if ((r = ssa_finish(ctx))) return r;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  st->picard_iterations = K;
  st->forward_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  ctx->adj_K = K;
  ctx->adj_every = every;
  ctx->adj_ready = true;
  return st->status;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

int ufe_ssa_adjoint_backward(ufe_ctx *ctx, const double *dJ_dU, const double *dJ_dV, double *g_logtau,
                             double *g_A, ufe_adjoint_stats *st) try {
  if (!ctx || !ctx->have_mesh || !dJ_dU || !dJ_dV || !g_logtau || !g_A || !st) return UFE_BAD_INPUT;
  if (!ctx->adj_ready) {
    ctx->err = "ufe_ssa_adjoint_backward needs a preceding ufe_ssa_adjoint_forward";
    return UFE_BAD_INPUT;
  }
  const int n = ctx->nA, nb = nblk(n), K = ctx->adj_K, every = ctx->adj_every;
  const ufe_linsolve_opts &L = ctx->adj_lin;
  const double omega = L.omega > 0.0 ? L.omega : ctx->params.SSA_SOR_omega;
  const int ks = L.precond_sweeps > 0 ? L.precond_sweeps : 2;
  struct GLGuard {
    ufe_ctx *c;
    ~GLGuard() { c->gl_active = false; }
  } gl_guard{ctx};
  ctx->gl_active = ctx->adj_gl;      // the rows the forward held fixed stay out of the adjoint solves
  const AaAcMesh am = aaac_mesh(ctx), mT = aaac_mesh_T(ctx);
  const ActiveRanges ar = active_ranges(ctx);
  int r;
  auto t0 = std::chrono::steady_clock::now();
  // The GL velocities P are the same in every iterate, so their adjoint pbar
  // collects: the adjoint of each iterate on those rows, and the coupling of
  // P into each step's free equations.  P is proportional to the rate factor of
  // the grounded vertex (calculate_GL_flux, :908-917), which turns pbar into a
  // contribution to dJ/dA at the end.
  if (ctx->adj_gl)
    k_fill<double2><<<nb, BLOCK, 0, ctx->stream>>>(ctx->adj_pbar, n, make_double2(0.0, 0.0));
  auto take_fixed = [&]() {
    if (ctx->adj_gl)
      k_take_skip_rows<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_skip, ctx->adj_g, ctx->adj_pbar);
  };
  // g_K = P^T dJ/du_K
  k_gather_perm_pair<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_perm, dJ_dU, ctx->adj_ubar, 0);
  k_gather_perm_pair<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_perm, dJ_dV, ctx->adj_ubar, 1);
  fold_T(ctx, ctx->adj_ubar);
  if ((r = copy_pair(ctx, ctx->adj_g, ctx->adj_ubar))) return r;
  take_fixed();
  k_fill<double><<<nb, BLOCK, 0, ctx->stream>>>(ctx->adj_gtau, n, 0.0);
  k_fill<double><<<nb, BLOCK, 0, ctx->stream>>>(ctx->adj_gA, n, 0.0);
  k_fill<double2><<<nb, BLOCK, 0, ctx->stream>>>(ctx->adj_lam, n, make_double2(0.0, 0.0));
  LAUNCHCHK(ctx);
  AdjPoint ap;
  ap.lam = ctx->adj_lam;
  ap.gtau = ctx->adj_gtau;
  ap.gA = ctx->adj_gA;
  ap.gux = ctx->adj_gs;
  ap.guy = ctx->adj_gs + n;
  ap.gvx = ctx->adj_gs + 2 * (size_t)n;
  ap.gvy = ctx->adj_gs + 3 * (size_t)n;
  ap.ubar = ctx->adj_ubar;
  const double2 *u_k = ctx->adj_uK;
  int seg_loaded = -1;
  for (int k = K; k >= 1; k--) {
    const int j = k - 1, s = j / every, off = j % every;
    const double2 *u_km1;
    if (off == 0) {
      u_km1 = ctx->adj_ck[s];
    } else {
      if (seg_loaded != s) {  // recompute the stored segment's inner iterates once
        if ((r = copy_pair(ctx, ctx->d_pair[0], ctx->adj_ck[s]))) return r;
        for (int i = 1; i < every && s * every + i <= K - 1; i++) {
          double rel = 0.0;
          int stt = 0;
          if ((r = adj_forward_step(ctx, &st->recompute_sweeps, &rel, &stt))) return r;
          if ((r = copy_pair(ctx, ctx->adj_seg[i - 1], ctx->d_pair[0]))) return r;
        }
        seg_loaded = s;
      }
      u_km1 = ctx->adj_seg[off - 1];
    }
    // eta, S, the system and the strain rates of step k, from u_{k-1}
    if ((r = copy_pair(ctx, ctx->d_pair[0], u_km1))) return r;
    if ((r = ssa_viscosity_rn(ctx, nullptr))) return r;
    if ((r = ssa_prepare_coeffs(ctx))) return r;
    double rel = 0.0;
    r = adj_solve(ctx, L.rel_tol, L.gmres_restart, ks, omega, L.max_sweeps, &st->adjoint_sweeps, &st->adjoint_matvecs,
                  &rel);
    st->max_adjoint_residual = std::max(st->max_adjoint_residual, rel);
    if (r == UFE_SOR_NOT_CONVERGED) st->status = UFE_SOR_NOT_CONVERGED;
    else if (r) return r;
    if (ctx->adj_gl) {                // pbar -= (A_free,fixed)^T lam
      apply_AT(ctx, mT, ar, ctx->adj_lam, ctx->adj_w, true);
      k_sub_skip_rows<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_skip, ctx->adj_w, ctx->adj_pbar);
    }
    ap.uk = u_k;
    ap.ukm1 = u_km1;
    k_adj_point<<<nb, BLOCK, 0, ctx->stream>>>(am, ssa_fields(ctx), ar, ap);
    k_adj_strain_T<<<nb, BLOCK, 0, ctx->stream>>>(mT, ar, ap.gux, ap.guy, ap.gvx, ap.gvy, ctx->adj_ubar);
    fold_T(ctx, ctx->adj_ubar);
    if ((r = copy_pair(ctx, ctx->adj_g, ctx->adj_ubar))) return r;
    take_fixed();
    LAUNCHCHK(ctx);
    u_k = u_km1;
  }
  if (ctx->adj_gl)
    k_gl_grad_A<<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), FI(ctx, "mask_gl_Ac"),
                                                            FI(ctx, "mask_sheet"), F(ctx, "A_flow_mean"),
                                                            F(ctx, "Ux_SSA_Ac"), F(ctx, "Uy_SSA_Ac"), ctx->d_iperm,
                                                            ctx->d_iAci, ctx->nCm, ctx->adj_pbar, ctx->adj_gA);
  // leave the forward's final velocities in place
  if ((r = copy_pair(ctx, ctx->d_pair[0], ctx->adj_uK))) return r;
  k_scatter_perm<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_perm, ctx->adj_gtau, g_logtau);
  k_scatter_perm<<<nb, BLOCK, 0, ctx->stream>>>(n, ctx->d_perm, ctx->adj_gA, g_A);
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  st->picard_iterations = K;
  st->backward_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return st->status;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}


// ---- batched ensembles -------------------------------------------------------
// (no reference counterpart: many independent linearised SSA systems, each
// src/ice_dynamics_module.f90:558-694, solved together)

int ufe_batch_define(ufe_ctx *ctx, int nmembers, const int32_t *nV, const int32_t *nAc) try {
  if (!ctx || nmembers < 0 || nmembers > 4096 || (nmembers > 0 && (!nV || !nAc))) return UFE_BAD_INPUT;
  ctx->b_nV.clear();
  ctx->b_nAc.clear();
  for (int b = 0; b < nmembers; b++) {
    if (nV[b] < 5 || nAc[b] < 1) {
      ctx->err = "every batch member needs at least 5 vertices and 1 Ac point";
      return UFE_BAD_INPUT;
    }
    ctx->b_nV.push_back(nV[b]);
    ctx->b_nAc.push_back(nAc[b]);
  }
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

static Chunks chunk_list(ufe_ctx *c) {
  Chunks ch;
  ch.n = c->n_chunk;
  ch.start = c->d_ch_start;
  ch.count = c->d_ch_count;
  ch.member = c->d_ch_member;
  return ch;
}

static int batch_alloc(ufe_ctx *ctx, int m, bool f32) {
  const int prec = f32 ? 1 : 0;
  if (ctx->bk_V && ctx->bk_m >= m && ctx->bk_prec == prec) return UFE_OK;
  const size_t n = ctx->nA, es = f32 ? sizeof(float2) : sizeof(double2);
  const size_t nb = ctx->nb;
  char *V, *Z, *w, *x, *R;
  int r;
  if ((r = dalloc(ctx, &V, es * n * (m + 1)))) return r;
  if ((r = dalloc(ctx, &Z, es * n * m))) return r;
  if ((r = dalloc(ctx, &w, es * n))) return r;
  if ((r = dalloc(ctx, &x, es * n))) return r;
  if ((r = dalloc(ctx, &R, es * n))) return r;
  ctx->bk_V = V;
  ctx->bk_Z = Z;
  ctx->bk_w = w;
  ctx->bk_x = x;
  ctx->bk_R = R;
  // zero the residual (its edge rows are never written) and the basis
  const int64_t nv = (int64_t)n * (m + 1);
  if (f32) {
    k_fill<float2><<<nblk(n), BLOCK, 0, ctx->stream>>>((float2 *)R, (int64_t)n, make_float2(0.0f, 0.0f));
    k_fill<float2><<<nblk(nv), BLOCK, 0, ctx->stream>>>((float2 *)V, nv, make_float2(0.0f, 0.0f));
  } else {
    k_fill<double2><<<nblk(n), BLOCK, 0, ctx->stream>>>((double2 *)R, (int64_t)n, make_double2(0.0, 0.0));
    k_fill<double2><<<nblk(nv), BLOCK, 0, ctx->stream>>>((double2 *)V, nv, make_double2(0.0, 0.0));
  }
  LAUNCHCHK(ctx);
  if (!ctx->bk_part) {
    if ((r = dalloc(ctx, &ctx->bk_part, (size_t)64 * ctx->n_chunk))) return r;
    if ((r = dalloc(ctx, &ctx->bk_H, nb * BHS))) return r;
    if ((r = dalloc(ctx, &ctx->bk_Hs, nb * BKS))) return r;
    if ((r = dalloc(ctx, &ctx->bk_y, nb * BKS))) return r;
    if ((r = dalloc(ctx, &ctx->bk_nrm, nb * BKS))) return r;
    if ((r = dalloc(ctx, &ctx->bk_scale, 2 * nb))) return r;
    if ((r = dalloc(ctx, &ctx->bk_rel, nb))) return r;
    if (!ctx->h_bk_rel) HIPCHK(ctx, hipHostMalloc((void **)&ctx->h_bk_rel, sizeof(double) * 4096));
  }
  ctx->bk_m = m;
  ctx->bk_prec = prec;
  if (ctx->bk_graph) (void)hipGraphExecDestroy(ctx->bk_graph);
  ctx->bk_graph = nullptr;
  return UFE_OK;
}

// residual of every member, its relative norm, and the scale of v0 = r/|r|
extern "C++" template <typename T>
static void batch_residual(ufe_ctx *ctx, double tol) {
  using T2 = typename V2T<T>::t;
  const AaAcMesh am = aaac_mesh(ctx);
  k_bresidual<T><<<ctx->n_chunk, BLOCK, 0, ctx->stream>>>(am, ctx->d_pair[0], ctx->d_pair[1], ctx->d_pair[2],
                                                         chunk_list(ctx), (T2 *)ctx->bk_R, ctx->bk_part);
  k_bdot_reduce<<<dim3(2, ctx->nb), 256, 0, ctx->stream>>>(ctx->d_mch_ptr, 2, ctx->bk_part, ctx->bk_nrm, BKS);
  k_bres_finish<<<nblk(ctx->nb), BLOCK, 0, ctx->stream>>>(ctx->nb, ctx->bk_nrm, tol, ctx->bk_rel,
                                                          ctx->bk_scale + ctx->nb, ctx->bk_scale);
}

// one GMRES(m) cycle of every member, then w += correction and the new residual
extern "C++" template <typename T>
static void batch_enqueue_cycle(ufe_ctx *ctx, int m, int ks, double omega, double tol) {
  using T2 = typename V2T<T>::t;
  const bool f32 = sizeof(T) == 4;
  const int n = ctx->nA, nb = nblk(n), NB = ctx->nb;
  const AaAcMesh am = aaac_mesh(ctx);
  const ActiveRanges ar = active_ranges(ctx);
  const Chunks ch = chunk_list(ctx);
  T2 *V = (T2 *)ctx->bk_V, *Z = (T2 *)ctx->bk_Z, *w = (T2 *)ctx->bk_w, *x = (T2 *)ctx->bk_x;
  double *beta = ctx->bk_scale + NB;
  k_bscale<T, T><<<nb, BLOCK, 0, ctx->stream>>>(n, (const T2 *)ctx->bk_R, ctx->bk_scale, ctx->d_mid, V);
  for (int j = 0; j < m; j++) {
    T2 *vj = V + (int64_t)j * n, *zj = Z + (int64_t)j * n;
    bool have_w = false;
    if (f32 && ctx->pc_amg) {
      have_w = amg_apply(ctx, am, (float)omega, (const float2 *)vj, (float2 *)zj, (float2 *)w);
    } else {
      k_fill<T2><<<nb, BLOCK, 0, ctx->stream>>>(zj, n, T2{T(0), T(0)});
      for (int k = 0; k < ks; k++) {
        const bool skip = k > 0 && !ctx->repeat_turn;
        const bool neu = !ctx->neumann_last || k == ks - 1;
        if (f32) enqueue_sweep_fp32(ctx, am, (float)omega, (float2 *)zj, (const float2 *)vj, k & 1, skip, neu);
        else enqueue_sweep_fp64_vec(ctx, am, omega, (double2 *)zj, (const double2 *)vj, k & 1, skip, neu);
      }
    }
    if (have_w) {
      // A z came with the post-smoothing
    } else if (f32)
      k_matvec<float><<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_cU32, ctx->d_Sxy32, ctx->d_EV32, ar,
                                                     (const float2 *)zj, (float2 *)w);
    else
      k_matvec<double><<<nb, BLOCK, 0, ctx->stream>>>(am, ctx->d_cU, ctx->d_Sxy, ctx->d_pair[1], ar,
                                                      (const double2 *)zj, (double2 *)w);
    double *hj = ctx->bk_H + (int64_t)j * 65;
    k_bdot<T><<<ctx->n_chunk, BLOCK, 0, ctx->stream>>>(ch, n, j + 1, V, w, ctx->bk_part);
    k_bdot_reduce<<<dim3(j + 1, NB), 256, 0, ctx->stream>>>(ctx->d_mch_ptr, j + 1, ctx->bk_part, hj, BHS);
    k_baxpy<T><<<nb, BLOCK, 0, ctx->stream>>>(n, j + 1, V, hj, BHS, ctx->d_mid, w);
    k_bdot<T><<<ctx->n_chunk, BLOCK, 0, ctx->stream>>>(ch, n, 1, w, w, ctx->bk_part);
    k_bdot_reduce<<<dim3(1, NB), 256, 0, ctx->stream>>>(ctx->d_mch_ptr, 1, ctx->bk_part, ctx->bk_nrm, BKS);
    k_bnorm_finish<<<nblk(NB), BLOCK, 0, ctx->stream>>>(NB, ctx->bk_nrm, ctx->bk_Hs + j, BKS, ctx->bk_rel, tol,
                                                        ctx->bk_scale);
    k_bscale<T, T><<<nb, BLOCK, 0, ctx->stream>>>(n, w, ctx->bk_scale, ctx->d_mid, V + (int64_t)(j + 1) * n);
  }
  k_blsq<<<NB, 64, 0, ctx->stream>>>(m, ctx->bk_H, ctx->bk_Hs, beta, ctx->bk_y);
  k_blincomb<T><<<nb, BLOCK, 0, ctx->stream>>>(n, m, Z, ctx->bk_y, ctx->d_mid, x);
  k_add_to_w<T><<<nb, BLOCK, 0, ctx->stream>>>(n, x, ctx->d_pair[0]);
  neumann_w(ctx);
  batch_residual<T>(ctx, tol);
}

static int batch_capture(ufe_ctx *ctx, bool f32, int m, int ks, double omega, double tol) {
  const int key = (f32 ? 1 : 2) + (ctx->pc_amg ? 4 * ctx->amg_nu : 0);   // precision and preconditioner
  if (ctx->bk_graph && ctx->bk_ks == ks && ctx->bk_omega == omega && ctx->bk_tol == tol &&
      ctx->bk_bs == ctx->tune_bs && ctx->bk_sched == ctx->tune_sched && ctx->bk_loads == ctx->tune_loads &&
      ctx->bk_m == m && ctx->bk_key == key)
    return UFE_OK;
  if (ctx->bk_graph) (void)hipGraphExecDestroy(ctx->bk_graph);
  ctx->bk_graph = nullptr;
  const bool prof = ctx->prof;
  ctx->prof = false;              // no event records inside the captured graph
  hipGraph_t g = nullptr;
  HIPCHK(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
  if (f32) batch_enqueue_cycle<float>(ctx, m, ks, omega, tol);
  else batch_enqueue_cycle<double>(ctx, m, ks, omega, tol);
  const hipError_t e1 = hipGetLastError();
  const hipError_t e2 = hipStreamEndCapture(ctx->stream, &g);
  ctx->prof = prof;
  if (e1 != hipSuccess || e2 != hipSuccess) {
    ctx->err = std::string("graph capture: ") + hipGetErrorString(e1 != hipSuccess ? e1 : e2);
    if (g) (void)hipGraphDestroy(g);
    return UFE_HIP_ERROR;
  }
  hipGraphExec_t ex = nullptr;
  const hipError_t e3 = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e3 != hipSuccess) {
    ctx->err = std::string("graph instantiate: ") + hipGetErrorString(e3);
    return UFE_HIP_ERROR;
  }
  ctx->bk_graph = ex;
  ctx->bk_key = key;
  ctx->bk_ks = ks;
  ctx->bk_omega = omega;
  ctx->bk_tol = tol;
  ctx->bk_bs = ctx->tune_bs;
  ctx->bk_sched = ctx->tune_sched;
  ctx->bk_loads = ctx->tune_loads;
  return UFE_OK;
}

int ufe_batch_linear_solve(ufe_ctx *ctx, const ufe_batch_opts *o, double *member_rel, ufe_batch_stats *st) try {
  if (!ctx || !ctx->have_mesh || !o || !st) return UFE_BAD_INPUT;
  std::memset(st, 0, sizeof(*st));
  if (ctx->nb == 0) {
    ctx->err = "no batch: call ufe_batch_define before ufe_mesh_upload";
    return UFE_BAD_INPUT;
  }
  if (o->gmres_restart < 1 || o->gmres_restart > 64 || !(o->rel_tol > 0.0) ||
      (o->precision != UFE_MIXED && o->precision != UFE_FP64)) {
    ctx->err = "ufe_batch_linear_solve: gmres_restart 1..64, rel_tol > 0, precision UFE_MIXED or UFE_FP64";
    return UFE_BAD_INPUT;
  }
  const bool f32 = o->precision == UFE_MIXED;
  if (o->precond_type != UFE_PRECOND_SOR && !(o->precond_type == UFE_PRECOND_MULTIGRID && f32)) {
    ctx->err = "ufe_batch_linear_solve: precond_type UFE_PRECOND_SOR, or UFE_PRECOND_MULTIGRID with UFE_MIXED";
    return UFE_BAD_INPUT;
  }
  ctx->pc_amg = o->precond_type == UFE_PRECOND_MULTIGRID;
  ctx->amg_nu = o->precond_sweeps > 0 ? o->precond_sweeps : 2;
  ctx->repeat_turn = false;          // batch preconditioner: turn colour once, Neumann at the end
  ctx->neumann_last = true;
  const int m = o->gmres_restart, ks = o->precond_sweeps > 0 ? o->precond_sweeps : 4;
  const double omega = o->omega > 0.0 ? o->omega : ctx->params.SSA_SOR_omega, tol = o->rel_tol;
  const int NB = ctx->nb;
  int r;
  if ((r = batch_alloc(ctx, m, f32))) return r;
  auto t0 = std::chrono::steady_clock::now();
  if (f32) k_to_f32_pair<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->nA, ctx->d_pair[1], ctx->d_EV32);
  if (ctx->pc_amg) {                  // the union of the members as one hierarchy
    ctx->amg_T = false;
    if ((r = amg_prepare(ctx))) return r;
    amg_refresh(ctx);
    LAUNCHCHK(ctx);
    if ((r = amg_capture(ctx))) return r;
  }
  if (ctx->n_neu) k_neumann_edges<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), ctx->d_pair[0], nullptr);
  k_neumann_scalar_pair_corners<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), ctx->d_pair[0]);
  if (f32) batch_residual<float>(ctx, tol);
  else batch_residual<double>(ctx, tol);
  LAUNCHCHK(ctx);
  if (o->use_graph && (r = batch_capture(ctx, f32, m, ks, omega, tol))) return r;
  const int max_cycles = o->max_cycles > 0 ? o->max_cycles : 100000;
  auto all_done = [&](double *worst, int *conv) {
    *worst = 0.0;
    *conv = 0;
    for (int b = 0; b < NB; b++) {
      *worst = std::max(*worst, ctx->h_bk_rel[b]);
      *conv += ctx->h_bk_rel[b] <= tol;
    }
    return *conv == NB;
  };
  double worst = 0.0;
  int conv = 0;
  int64_t cpass = 0;
  while (true) {
    HIPCHK(ctx, hipMemcpyAsync(ctx->h_bk_rel, ctx->bk_rel, sizeof(double) * NB, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    if (all_done(&worst, &conv) || st->cycles >= max_cycles || !std::isfinite(worst)) break;
    if (o->use_graph) {
      HIPCHK(ctx, hipGraphLaunch(ctx->bk_graph, ctx->stream));
    } else {
      if (f32) batch_enqueue_cycle<float>(ctx, m, ks, omega, tol);
      else batch_enqueue_cycle<double>(ctx, m, ks, omega, tol);
      LAUNCHCHK(ctx);
    }
    st->cycles++;
    cpass += (int64_t)m * (ctx->pc_amg ? amg_passes(ctx) : precond_passes(ctx, ks));
    st->sweeps = (int32_t)(cpass / 5);
  }
  st->converged = conv;
  st->max_rel_residual = worst;
  st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  st->status = conv == NB ? UFE_OK : UFE_SOR_NOT_CONVERGED;
  if (member_rel) std::memcpy(member_rel, ctx->h_bk_rel, sizeof(double) * NB);
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

int ufe_batch_solve_SSA(ufe_ctx *ctx, int picard_iterations, const ufe_batch_opts *o, double *member_rel,
                        ufe_batch_stats *st) try {
  if (!ctx || !ctx->have_mesh || !o || !st || picard_iterations < 1) return UFE_BAD_INPUT;
  if (ctx->nb == 0) {
    ctx->err = "no batch: call ufe_batch_define before ufe_mesh_upload";
    return UFE_BAD_INPUT;
  }
  ufe_batch_stats tot{};
  auto t0 = std::chrono::steady_clock::now();
  int r;
  if ((r = ssa_gather(ctx))) return r;
  for (int k = 0; k < picard_iterations; k++) {
    if ((r = ssa_viscosity_rn(ctx, nullptr))) return r;
    if ((r = ssa_prepare_coeffs(ctx))) return r;
    ufe_batch_stats s1;
    if ((r = ufe_batch_linear_solve(ctx, o, member_rel, &s1))) return r;
    tot.cycles += s1.cycles;
    tot.sweeps += s1.sweeps;
    tot.converged = s1.converged;
    tot.max_rel_residual = s1.max_rel_residual;
    if (s1.status != UFE_OK) tot.status = s1.status;
  }
  if ((r = ssa_finish(ctx))) return r;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  tot.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  *st = tot;
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

// Time `sweeps` FP32 sweeps (colour passes plus Neumann) of the uploaded mesh
// (a single mesh or a batch) for every launch shape and keep the fastest.
int ufe_sweep_autotune(ufe_ctx *ctx, int sweeps, ufe_sweep_tuning *out) try {
  if (!ctx || !ctx->have_mesh || !out || sweeps < 1) return UFE_BAD_INPUT;
  std::memset(out, 0, sizeof(*out));
  const AaAcMesh am = aaac_mesh(ctx);
  k_to_f32_pair<<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->nA, ctx->d_pair[1], ctx->d_EV32);
  LAUNCHCHK(ctx);
  const bool prof = ctx->prof;
  ctx->prof = false;
  const int bss[4] = {64, 128, 256, 512};
  hipEvent_t a, b;
  HIPCHK(ctx, hipEventCreate(&a));
  HIPCHK(ctx, hipEventCreate(&b));
  double best = HUGE_VAL;
  int nbest = 256, sbest = 0, lbest = 0, k = 0;
  for (int loads = 0; loads < 4; loads++)
    for (int bs : bss)
      for (int sched = 0; sched < 2; sched++) {
        ctx->tune_bs = bs;
        ctx->tune_sched = sched;
        ctx->tune_loads = loads;
        enqueue_sweep_fp32(ctx, am, 1.0f, ctx->d_D32, ctx->d_R32, false);  // warm-up
        (void)hipEventRecord(a, ctx->stream);
        for (int i = 0; i < sweeps; i++) enqueue_sweep_fp32(ctx, am, 1.0f, ctx->d_D32, ctx->d_R32, i & 1);
        (void)hipEventRecord(b, ctx->stream);
        LAUNCHCHK(ctx);
        HIPCHK(ctx, hipEventSynchronize(b));
        float ms = 0.0f;
        HIPCHK(ctx, hipEventElapsedTime(&ms, a, b));
        const double us = 1e3 * ms / sweeps;
        out->cand_threads[k] = bs;
        out->cand_schedule[k] = sched;
        out->cand_loads[k] = loads;
        out->cand_us_per_sweep[k] = us;
        k++;
        if (us < best) {
          best = us;
          nbest = bs;
          sbest = sched;
          lbest = loads;
        }
      }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  ctx->prof = prof;
  // the sweeps above ran on scratch vectors: clear the correction again
  k_fill<float2><<<nblk(ctx->nA), BLOCK, 0, ctx->stream>>>(ctx->d_D32, ctx->nA, make_float2(0.0f, 0.0f));
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  out->n_candidates = k;
  out->threads_per_block = nbest;
  out->schedule = sbest;
  out->loads = lbest;
  ctx->tune_bs = nbest;
  ctx->tune_sched = sbest;
  ctx->tune_loads = lbest;
  return UFE_OK;
} catch (const std::exception &e) {
  return host_failure(ctx, e.what());
} catch (...) {
  return host_failure(ctx, "unknown exception");
}

int ufe_sweep_tuning_set(ufe_ctx *ctx, int threads_per_block, int schedule, int loads) {
  if (!ctx || (threads_per_block != 64 && threads_per_block != 128 && threads_per_block != 256 &&
               threads_per_block != 512) || schedule < 0 || schedule > 1 || loads < 0 || loads > 3)
    return UFE_BAD_INPUT;
  ctx->tune_bs = threads_per_block;
  ctx->tune_sched = schedule;
  ctx->tune_loads = loads;
  return UFE_OK;
}

int ufe_profile_enable(ufe_ctx *ctx, int enable) {
  if (!ctx) return UFE_BAD_INPUT;
  ctx->prof = enable != 0;
  return UFE_OK;
}
int ufe_profile_read(ufe_ctx *ctx, ufe_kernel_profile *out) {
  if (!ctx || !out) return UFE_BAD_INPUT;
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  prof_collect(ctx);
  *out = ctx->prof_acc;
  ctx->prof_acc = ufe_kernel_profile{};
  return UFE_OK;
}
int ufe_sweep_bytes(ufe_ctx *ctx, double *b64, double *b32, double *mean_deg, int64_t *rows) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  double s64 = 0.0, s32 = 0.0;
  int64_t n = 0;
  for (int c = 0; c < 5; c++) {
    s64 += ctx->bytes64[c];
    s32 += ctx->bytes32[c];
    n += ctx->colour_active[c];
  }
  if (b64) *b64 = s64;
  if (b32) *b32 = s32;
  if (mean_deg) *mean_deg = n ? ctx->degsum / (double)n : 0.0;
  if (rows) *rows = n;
  return UFE_OK;
}

int ufe_field_fill(ufe_ctx *ctx, int id, double value) {
  if (!ctx || !ctx->have_mesh || id < 0 || id >= NFIELDS) return UFE_BAD_INPUT;
  const FieldDef &fd = FIELDS[id];
  const int64_t n = (int64_t)grid_len(ctx, fd.grid);
  if (fd.pair >= 0) {
    // fill one component of an interleaved pair
    k_fill_pair_comp<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, ctx->d_pair[fd.pair], fd.comp, value);
  } else if (fd.dtype == D_F64) {
    k_fill<double><<<nblk(n), BLOCK, 0, ctx->stream>>>((double *)ctx->field_ptr[id], n, value);
  } else {
    k_fill<int32_t><<<nblk(n), BLOCK, 0, ctx->stream>>>((int32_t *)ctx->field_ptr[id], n, (int32_t)value);
  }
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

// ---- calculate_ice_thickness_change -----------------------------------------
int ufe_calculate_ice_thickness_change(ufe_ctx *ctx, double dt) {
  if (!ctx || !ctx->have_mesh) return UFE_BAD_INPUT;
  double *dVi = F(ctx, "dVi_in");
  k_fill<double><<<nblk((int64_t)ctx->nV * ctx->nCm), BLOCK, 0, ctx->stream>>>(dVi, (int64_t)ctx->nV * ctx->nCm, 0.0);
  k_mc_flux<<<nblk(ctx->nAc), BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), F(ctx, "Hi"), F(ctx, "Up_SIA_Ac"),
                                                         F(ctx, "Up_SSA_Ac"), ctx->d_Cw, dt, dVi);
  AaMesh am = aa_mesh(ctx);
  k_mc_rescale<<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(am, F(ctx, "Hi"), F(ctx, "SMB_year"), F(ctx, "BMB"), dt,
                                                           dVi, ctx->d_ViSMB);
  k_mc_update<<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(am, dVi, ctx->d_ViSMB, dt, FI(ctx, "mask_noice"),
                                                          F(ctx, "dHi_dt"), F(ctx, "Hi"), F(ctx, "Hi_prev"),
                                                          ctx->params.zero_Hi_at_edges);
  LAUNCHCHK(ctx);
  HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  return UFE_OK;
}

// ---- operators -------------------------------------------------------------
#define NEED_MESH(ctx) \
  if (!(ctx) || !(ctx)->have_mesh) return UFE_BAD_INPUT

int ufe_op_derivatives_Aa(ufe_ctx *ctx, const double *d, double *ddx, double *ddy) {
  NEED_MESH(ctx);
  k_deriv_Aa<<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(aa_mesh(ctx), d, ddx, ddy);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_curvatures_Aa(ufe_ctx *ctx, const double *d, double *a, double *b, double *c) {
  NEED_MESH(ctx);
  k_curv_Aa<<<nblk(ctx->nV), BLOCK, 0, ctx->stream>>>(aa_mesh(ctx), d, a, b, c);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_derivatives_Aa_3D(ufe_ctx *ctx, const double *d, double *ddx, double *ddy, int nz) {
  NEED_MESH(ctx);
  layered(ctx->nV, nz, 1, [&](auto G, dim3 grid) {
    k_deriv_Aa_3D<G.value><<<grid, BLOCK, 0, ctx->stream>>>(aa_mesh(ctx), nz, d, ddx, ddy);
  });
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_neumann_Aa(ufe_ctx *ctx, double *d) { return ufe_op_neumann_Aa_3D(ctx, d, 1); }
int ufe_op_neumann_Aa_3D(ufe_ctx *ctx, double *d, int nz) {
  NEED_MESH(ctx);
  neumann_Aa(ctx, nz, d);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_upwind_derivatives_3D(ufe_ctx *ctx, const double *U, const double *V, const double *d, double *ddx,
                                 double *ddy, int nz, int *missing) {
  NEED_MESH(ctx);
  if (!U || !V || !d || !ddx || !ddy || nz < 1) return UFE_BAD_INPUT;
  hipStream_t q = ctx->stream;
  HIPCHK(ctx, hipMemsetAsync(ctx->d_icount, 0, sizeof(int32_t), q));
  layered(ctx->nV, nz, 1, [&](auto G, dim3 grid) {
    k_upwind_3D<G.value><<<grid, BLOCK, 0, q>>>(aa_mesh(ctx), tri_mesh(ctx), nz, U, V, d, ddx, ddy, ctx->d_icount);
  });
  LAUNCHCHK(ctx);
  int32_t h = 0;
  HIPCHK(ctx, hipMemcpyAsync(&h, ctx->d_icount, sizeof(int32_t), hipMemcpyDeviceToHost, q));
  HIPCHK(ctx, hipStreamSynchronize(q));
  if (missing) *missing = h;
  return UFE_OK;
}
int ufe_op_derivatives_Ac(ufe_ctx *ctx, const double *d, double *ddx, double *ddy, double *ddp, double *ddo) {
  NEED_MESH(ctx);
  k_deriv_Ac<<<nblk(ctx->nAc), BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), d, ddx, ddy, ddp, ddo);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_derivatives_AaAc(ufe_ctx *ctx, const double *d, double *ddx, double *ddy) {
  NEED_MESH(ctx);
  const int n = ctx->nA;
  k_gather_perm<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, ctx->d_perm, d, ctx->d_tmp[0]);
  k_deriv_AaAc<<<xcd_grid(n), BLOCK, 0, ctx->stream>>>(aaac_mesh(ctx), ctx->d_perm, ctx->d_tmp[0], ddx, ddy);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_curvatures_AaAc(ufe_ctx *ctx, const double *d, double *a, double *b, double *c) {
  NEED_MESH(ctx);
  const int n = ctx->nA;
  k_gather_perm<<<nblk(n), BLOCK, 0, ctx->stream>>>(n, ctx->d_perm, d, ctx->d_tmp[0]);
  k_curv_AaAc<<<nblk(n), BLOCK, 0, ctx->stream>>>(aaac_mesh(ctx), ctx->d_perm, ctx->d_tmp[0], a, b, c);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_neumann_AaAc(ufe_ctx *ctx, double *d) {
  NEED_MESH(ctx);
  if (ctx->n_neu)
    k_neumann_scalar<<<nblk(ctx->n_neu), BLOCK, 0, ctx->stream>>>(neu_list(ctx), ctx->d_perm, d);
  if (ctx->n_cor)                    // a batch need not have corner codes
    k_neumann_scalar<<<nblk(ctx->n_cor, 64), 64, 0, ctx->stream>>>(cor_list(ctx), ctx->d_perm, d);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_map_Aa_to_Ac(ufe_ctx *ctx, const double *a, double *b) { return ufe_op_map_Aa_to_Ac_3D(ctx, a, b, 1); }
int ufe_op_map_Aa_to_Ac_3D(ufe_ctx *ctx, const double *a, double *b, int nz) {
  NEED_MESH(ctx);
  layered(ctx->nAc, nz, 1, [&](auto G, dim3 grid) {
    k_map_Aa_to_Ac<G.value><<<grid, BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), nz, a, b);
  });
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_map_Ac_to_Aa(ufe_ctx *ctx, const double *a, double *b) { return ufe_op_map_Ac_to_Aa_3D(ctx, a, b, 1); }
int ufe_op_map_Ac_to_Aa_3D(ufe_ctx *ctx, const double *a, double *b, int nz) {
  NEED_MESH(ctx);
  k_map_Ac_to_Aa<<<layer_grid(ctx->nV, nz, 1), BLOCK, 0, ctx->stream>>>(aa_mesh(ctx), ctx->nAc, nz, a, b);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}
int ufe_op_rotate_xy_to_po(ufe_ctx *ctx, const double *x, const double *y, double *p, double *o) {
  NEED_MESH(ctx);
  k_rotate<<<nblk(ctx->nAc), BLOCK, 0, ctx->stream>>>(ac_mesh(ctx), x, y, p, o);
  LAUNCHCHK(ctx);
  return ufe_synchronize(ctx);
}

}  // extern "C"
