// HIP engine behind the mjmlx C API: gfx950 kernels and the batched sim.
//
// One 64-lane wavefront steps one env: the env's state and every per-step
// intermediate live in that workgroup's LDS workspace (kernels.h), state is
// read from HBM once per call and written back once after all substeps.
// One workgroup per env: the hardware dispatcher refills CUs as envs finish.
// The step kernels themselves are built per narrow-phase set in step_np.hip.
//
// Replaces the reference's per-stage Vulkan dispatches and the host substep
// loop (reference src/batched.cpp:980-1228,1469-1504).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <memory>
#include <mutex>
#include <sstream>
#include <stdexcept>
#include <string>
#include <vector>

#include "hostmodel.h"
#include "kernels.h"
#include "mjmlx/mjmlx_hip.h"
#include "mlp.h"
#include "step_launch.h"

namespace {

#define HIPOK(expr)                                                                           \
  do {                                                                                        \
    hipError_t e_ = (expr);                                                                   \
    if (e_ != hipSuccess) {                                                                   \
      throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e_) + " at " + \
                               __FILE__ + ":" + std::to_string(__LINE__) + " (" #expr ")");  \
    }                                                                                         \
  } while (0)

void report(const char* fn, const std::exception& e) { std::fprintf(stderr, "%s error: %s\n", fn, e.what()); }

}  // namespace

// ------------------------------------------------------------------ kernels
// mj_ray for every (env, ray): one wave per env computes the env's geom
// poses in its workspace, its lanes take the rays (reference
// src/batched.cpp:1808-1893)
template <int GWS>
__global__ void __launch_bounds__(64) k_raycast(mjk::DModel m, mjk::Layout L, const float* qpos, const float* rand,
                                                int nrand, const float* pnt, const float* vec, int nray,
                                                const int* gmask, float* dist, int* gid, int B, float* gws) {
  extern __shared__ __align__(16) float lds[];
  int env = blockIdx.x;
  if (env >= B) return;
  float* w = GWS ? gws + (size_t)env * L.total : lds;
  mjk::run_rays(m, L, w, qpos, rand, nrand, pnt, vec, nray, gmask, dist, gid, env);
}

// sprev: accelerometer state [B][pstride] whose last entry (previous velocity
// valid) a reset clears, or null
__global__ void k_reset(const int* mask, float* qpos, float* qvel, float* qws, const float* qpos0, int B, int nq, int nv,
                        float* sprev, int pstride) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= B || !mask[e]) return;
  if (sprev) sprev[(size_t)e * pstride + pstride - 1] = 0.f;
  for (int i = 0; i < nq; i++) qpos[(size_t)e * nq + i] = qpos0[i];
  for (int i = 0; i < nv; i++) { qvel[(size_t)e * nv + i] = 0.f; qws[(size_t)e * nv + i] = 0.f; }
}

// Launch order of the step's workgroups: envs by decreasing solver iterations
// of the previous call (a counting sort on min(niter, ORDER_KEYS - 1), one
// workgroup), so the envs that ran longest start first and the launch ends
// on short ones. Envs of equal count keep no particular order: each env's
// result does not depend on when it runs.
constexpr int ORDER_KEYS = 128;
__global__ void __launch_bounds__(1024) k_order(const int* __restrict__ niter, int* __restrict__ order, int B) {
  __shared__ int start[ORDER_KEYS];
  int t = (int)threadIdx.x;
  if (t < ORDER_KEYS) start[t] = 0;
  __syncthreads();
  auto key = [&](int e) {  // bucket 0 holds the longest envs
    int k = niter[e];
    k = k < 0 ? 0 : (k > ORDER_KEYS - 1 ? ORDER_KEYS - 1 : k);
    return ORDER_KEYS - 1 - k;
  };
  for (int e = t; e < B; e += (int)blockDim.x) atomicAdd(&start[key(e)], 1);
  __syncthreads();
  if (t == 0) {
    int acc = 0;
    for (int k = 0; k < ORDER_KEYS; k++) { int c = start[k]; start[k] = acc; acc += c; }
  }
  __syncthreads();
  for (int e = t; e < B; e += (int)blockDim.x) order[atomicAdd(&start[key(e)], 1)] = e;
}

// packed readback: [qpos, qvel, |cfrc_ext force| of chosen bodies, sum sq and sum abs of qfrc_actuator range]
// (reference src/batched.cpp:1683-1708)
__global__ void k_pack(const float* qpos, const float* qvel, const float* cfrc, const float* qfa, const int* bodies,
                       int nsel, int dof_lo, int ndof, int B, int nq, int nv, int nb, float* out) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= B) return;
  int stride = nq + nv + nsel + 2;
  float* o = out + (size_t)e * stride;
  for (int i = 0; i < nq; i++) o[i] = qpos[(size_t)e * nq + i];
  for (int i = 0; i < nv; i++) o[nq + i] = qvel[(size_t)e * nv + i];
  for (int k = 0; k < nsel; k++) {
    const float* f = cfrc + ((size_t)e * nb + bodies[k]) * 6 + 3;
    o[nq + nv + k] = sqrtf(f[0] * f[0] + f[1] * f[1] + f[2] * f[2]);
  }
  float sq = 0.f, ab = 0.f;
  for (int k = 0; k < ndof; k++) { float t = qfa[(size_t)e * nv + dof_lo + k]; sq += t * t; ab += fabsf(t); }
  o[nq + nv + nsel] = sq;
  o[nq + nv + nsel + 1] = ab;
}

// ------------------------------------------------------------------ handles
struct MjmlxModel {
  mjh::Model m;
  mjh::LoadOptions opt;
};

struct MjmlxData {
  int unused;
};

enum { RAYS_ONE_COPY = 256 << 10 };
struct MjmlxBatchedSim {
  mjh::Model model;
  mjh::Blob blob;
  mjk::DModel dm;
  mjk::Layout L;
  std::vector<mjh::LayoutField> fields;
  int B = 0, nq = 0, nv = 0, nu = 0, nb = 0;
  size_t lds_bytes = 0;
  char* d_blob = nullptr;
  float *d_qpos = nullptr, *d_qvel = nullptr, *d_qws = nullptr, *d_ctrl = nullptr, *d_qpos0 = nullptr;
  int *d_niter = nullptr, *d_status = nullptr, *d_ncon = nullptr, *d_nefc = nullptr, *d_queue = nullptr, *d_mask = nullptr;
  int* d_order = nullptr;  // workgroup slot -> env of the fused step launch (k_order)
  int* d_ident = nullptr;  // the identity order of every other launch
  // longest envs first (k_order), for batches of at least 16 envs per CU:
  // smaller ones (the boxes workload's groups, ~565 envs on concurrent
  // streams) lose more to the sort's launch than the shorter tail saves.
  // MJMLX_HIP_ORDER=0/1 forces it off / on.
  int order_mode = -1;
  float* d_aux[7] = {};  // xpos xquat subtree_com cinert cvel qfrc_actuator cfrc_ext
  float* h_aux[7] = {};
  bool aux_on = false;
  float *h_qpos = nullptr, *h_qvel = nullptr, *h_ctrl = nullptr;
  int* h_mask = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr, ev_ctrl = nullptr;
  bool timed = false, ctrl_pending = false;
  int persistent = 0, grid = 0, ncu = 0;
  int npset = 0;  // narrow-phase set compiled into the step kernel
  float* d_gws = nullptr;  // per-env workspaces in device memory when they exceed the LDS of a workgroup
  mjk::KParams* d_kp = nullptr;  // device copy of dm and L, which the step kernels read
  // LDS workspaces with room for fewer contacts than the model's capacity, for
  // the envs that fit them (try_compact), and the marks of those that do not
  bool compact = false;
  int compact_variant = 0;
  mjk::Layout Lc;
  mjk::KParams* d_kpc = nullptr;
  int* d_redo = nullptr;
  bool ctrl_zero = true;   // d_ctrl holds zeros (set at creation; cleared by an upload)
  bool use_gws = false;    // launch the device-memory workspace variant
  bool lds_ok = false;     // the workspace fits the LDS of a workgroup
  bool high_occ = false;   // LDS admits more than 8 envs per CU: the 168-VGPR kernel
  bool big_regs = false;   // LDS admits at most 4 envs per CU: the 512-register kernel
  bool half = false;       // 32 lanes per env, two envs per wave (LDS workspaces only)
  bool half_ok = false;    // the model fits the 32-lane kernels (at most 32 dofs, two workspaces per workgroup)
  int ws_mode = 0;
  // learned control step captured as a HIP graph (mjmlx_batched_set_graph):
  // the captured launch sequence and the inputs it was captured for
  bool graph_on = false;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  int g_n = -1, g_cur = -1, g_mode = -1;
  const void *g_mlp = nullptr, *g_xb = nullptr;
  bool g_gws = false, g_occ = false, g_big = false, g_half = false, g_compact = false;
  // packed readback
  int* d_pack_bodies = nullptr;
  float* d_pack = nullptr;
  int pack_nsel = 0, pack_lo = 0, pack_ndof = 0, pack_stride = -1;
  // learned warm start: raw features after each substep (double-buffered) and predictions
  MjmlxMLP* mlp = nullptr;
  float* d_feat[2] = {};
  float* d_pred = nullptr;
  int feat_cur = 0;
  bool feat_valid = false;
  int feat_mode = 0;  // 1: features end with the previous substep's qacc and the network predicts the change
  int nfeat() const { return dm.nfeat + (feat_mode ? nv : 0); }
  // domain randomisation: per-env parameter blocks (mjk::rand_size floats per
  // env, env-major), the host copy the setters edit, and the free-joint count
  float* d_rand = nullptr;
  std::vector<float> h_rand;
  int nrand = 0, nfree = 0;
  // sensors: sensordata [B][nsensordata] (device and a pinned host copy) and
  // the accelerometers' previous frame velocities [B][3 * nacc + 1]
  float *d_sensordata = nullptr, *h_sensordata = nullptr, *d_sens_prev = nullptr;
  // raycast buffers: points and directions [2][B][nray][3], results, geom filter (grown on demand)
  float *d_rays = nullptr, *d_rdist = nullptr;
  int *d_rgid = nullptr, *d_gmask = nullptr;
  size_t ray_cap = 0;
  std::vector<float> h_rays;  // both arrays of a small scan (at most RAYS_ONE_COPY bytes)
  // scratch host buffers for dumps
  float *d_dump1 = nullptr, *d_dump2 = nullptr;
  size_t dump_cap = 0;

  size_t aux_len(int i) const {
    static const int per[7] = {3, 4, 3, 10, 6, 0, 6};
    return i == 5 ? (size_t)B * nv : (size_t)B * nb * per[i];
  }
};

namespace {

void free_sim(MjmlxBatchedSim* s) {
  if (!s) return;
  if (s->stream) hipStreamSynchronize(s->stream);
  void* dev[] = {s->d_blob, s->d_qpos, s->d_qvel, s->d_qws, s->d_ctrl, s->d_qpos0, s->d_niter, s->d_status,
                 s->d_ncon, s->d_nefc, s->d_queue, s->d_mask, s->d_pack_bodies, s->d_pack, s->d_dump1, s->d_dump2,
                 s->d_feat[0], s->d_feat[1], s->d_pred, s->d_gws, s->d_rand, s->d_rays, s->d_rdist,
                 s->d_rgid, s->d_gmask, s->d_sensordata, s->d_sens_prev, s->d_kp, s->d_kpc, s->d_redo, s->d_order,
                 s->d_ident};
  for (void* p : dev) if (p) hipFree(p);
  for (int i = 0; i < 7; i++) { if (s->d_aux[i]) hipFree(s->d_aux[i]); if (s->h_aux[i]) hipHostFree(s->h_aux[i]); }
  if (s->h_qpos) hipHostFree(s->h_qpos);
  if (s->h_qvel) hipHostFree(s->h_qvel);
  if (s->h_ctrl) hipHostFree(s->h_ctrl);
  if (s->h_mask) hipHostFree(s->h_mask);
  if (s->h_sensordata) hipHostFree(s->h_sensordata);
  if (s->ev0) hipEventDestroy(s->ev0);
  if (s->ev1) hipEventDestroy(s->ev1);
  if (s->ev_ctrl) hipEventDestroy(s->ev_ctrl);
  if (s->gexec) hipGraphExecDestroy(s->gexec);
  if (s->graph) hipGraphDestroy(s->graph);
  if (s->stream) hipStreamDestroy(s->stream);
  delete s;
}

// dm and L to the device copy the step kernels read, once the steps queued
// before have read the previous contents
void upload_kparams(MjmlxBatchedSim* s) {
  mjk::KParams kp{s->dm, s->L};
  HIPOK(hipStreamSynchronize(s->stream));
  HIPOK(hipMemcpy(s->d_kp, &kp, sizeof kp, hipMemcpyHostToDevice));
  if (s->d_kpc) {
    kp.L = s->Lc;
    HIPOK(hipMemcpy(s->d_kpc, &kp, sizeof kp, hipMemcpyHostToDevice));
  }
}

// Smaller LDS workspaces for a big model's usual contact counts. A model's
// contact capacity is sized for its pairs' maxima (8 free boxes: 144 contacts,
// 576 rows, 100 KB: one env per CU and a batch of 1000 in four rounds; beyond 9
// boxes it does not fit LDS at all), while landed boxes keep 3.5-4 contacts a
// body. When the whole batch can be resident at once with room for 5 contacts
// per free body, the step first runs with that capacity, and the few envs that
// need more are stepped again, from the state they were in, by the full-size
// kernel. One round in LDS takes 1 / 1.45 of the device-memory time (18 boxes,
// 250 envs: 2.30 against 3.22 ms per control step), two take longer, so it is
// used only where one round holds the batch. 8 boxes, 1000 envs: 4.9 -> 1.35 ms.
// Results do not depend on which launch stepped an env.
// try_compact: whether small workspaces were set up.
bool try_compact(MjmlxBatchedSim* s, const mjh::Caps& caps, const std::vector<mjh::CollisionPair>& pairs,
                 size_t lds_cu, size_t lds_max, size_t per_cu) {
  const auto& m = s->model;
  // the accelerometers' history is written every substep: an env cannot be stepped twice
  if (m.nsensor > 0 || s->blob.proto.jw <= 0 || per_cu > 8) return false;
  size_t budget = std::min({lds_cu / per_cu / 1280 * 1280, lds_max});  // LDS is given out in 1280-byte pieces
  int rpc = 1, fixed = 0;
  for (auto& p : pairs)
    rpc = std::max(rpc, p.condim == 1 ? 1 : (m.cone == mjh::CONE_PYRAMIDAL ? 2 * (p.condim - 1) : p.condim));
  for (int k = 0; k < m.nv; k++) fixed += m.dof_frictionloss[k] > 0;
  for (int j = 0; j < m.njnt; j++) fixed += m.jnt_limited[j] ? 2 : 0;
  auto layout = [&](int c) {
    mjk::Layout l = mjk::make_layout(m.nq, m.nv, m.nu, m.nbody, m.njnt, m.ngeom, c, std::min(caps.maxefc, fixed + rpc * c),
                                     m.solver == mjh::SOL_NEWTON, s->nrand, s->blob.proto.jw, s->blob.proto.nM);
    l.efc_cap = caps.efc_cap;
    l.con_cap = caps.con_cap;
    return l;
  };
  int lo = std::min(caps.maxcon, std::max(16, 5 * s->nfree)), hi = caps.maxcon;
  if (layout(lo).total * sizeof(float) > budget) return false;
  while (lo < hi) {
    int c = (lo + hi + 1) / 2;
    if (layout(c).total * sizeof(float) <= budget) lo = c;
    else hi = c - 1;
  }
  s->Lc = layout(lo);
  HIPOK(hipMalloc(&s->d_kpc, sizeof(mjk::KParams)));
  HIPOK(hipMalloc(&s->d_redo, (size_t)s->B * sizeof(int)));
  s->compact = true;
  // register budget by the envs LDS admits per CU, as for full workspaces
  s->compact_variant = lds_cu / (s->Lc.total * sizeof(float)) <= 4 ? mjk::VAR_LDS_BIG : mjk::VAR_LDS;
  return true;
}
// Placement of a model of more than SPARSE_ROWS_NV dofs whose batch is not one
// LDS round; `fits`: each env's full workspace alone fits LDS. ms per control
// step, LDS rounds at full size / small workspaces / device memory:
//   free bodies (6-9 boxes, CG and Newton, 600-4096 envs; landing): 6 boxes, 600
//   envs 1.95 / 1.13 / 1.50; 8, 600 2.93 / 1.09 / 1.47; 8, 4096 15.7 / - / 3.8;
//   Newton 6, 1100 2.42 / 1.17 / 1.73; 8, 2100 15.2 / - / 6.4. Small workspaces,
//   else device memory, which two LDS rounds never beat.
//   articulated, pyramidal cones, Newton or CG: small workspaces win (two
//   quadrupeds, 36 dofs, 1100 envs 0.99 / 0.61 / 0.97, standing 1.93 / 1.70 /
//   2.56; a 54-dof tree, 300 envs 2.90 / 1.73 / 2.54). Device memory holds 8
//   envs per CU and is up to 1.55 times slower a round: with three LDS rounds to
//   one or two standing quadrupeds lose (three of them, 1100 envs 4.38 / - / 5.16;
//   two, 2100 envs 2.73 / - / 3.07; a 40-dof chain, 2100 envs 3.31 / - / 3.80),
//   from four times its rounds all gain (three quadrupeds, 4096 envs 6.2 / - /
//   4.5; the tree, 1100 envs 10.6 / - / 5.9; a 66-dof scene 8.0 / - / 7.4).
//   articulated with elliptic cones under Newton: H is factored in the workspace
//   at every step; no batch of them was measured to gain. They stay in LDS.
// A workspace set in device memory that cannot be allocated goes back to LDS.
void place_big(MjmlxBatchedSim* s, const mjh::Caps& caps, const std::vector<mjh::CollisionPair>& pairs, size_t lds_cu,
               size_t lds_max) {
  const auto& m = s->model;
  if (s->nv <= mjk::SPARSE_ROWS_NV) return;
  // explicit capacities, row forms and placements are kept as given
  for (const char* v : {"MJMLX_HIP_MAXCON", "MJMLX_HIP_MAXEFC", "MJMLX_HIP_LDS_MAX", "MJMLX_HIP_GLOBAL_WORKSPACE",
                        "MJMLX_HIP_HIGH_OCC", "MJMLX_HIP_BIG_REGS", "MJMLX_HIP_REF_CAPS", "MJMLX_MAX_EFC",
                        "MJMLX_HIP_DENSE_ROWS"})
    if (std::getenv(v)) return;
  size_t per_cu = ((size_t)s->B + s->ncu - 1) / std::max(1, s->ncu);
  bool fits = !s->use_gws, free_bodies = 6 * s->nfree == s->nv;
  if (fits && lds_cu / s->lds_bytes >= per_cu) return;  // one round already
  if (!free_bodies && m.solver == mjh::SOL_NEWTON && m.cone != mjh::CONE_PYRAMIDAL) return;
  if (try_compact(s, caps, pairs, lds_cu, lds_max, per_cu) || !fits) return;
  size_t in_lds = lds_cu / s->lds_bytes, lds_rounds = (per_cu + in_lds - 1) / in_lds;
  if (!free_bodies && lds_rounds < 4 * ((per_cu + 7) / 8)) return;
  if (hipMalloc(&s->d_gws, (size_t)s->B * s->L.total * sizeof(float)) != hipSuccess) {
    (void)hipGetLastError();
    s->d_gws = nullptr;
    return;
  }
  s->use_gws = true;
  s->high_occ = s->big_regs = false;
}

// the autotuner's number of small LDS workspaces with a full-size rerun
// (try_compact); 0 .. VAR_N - 1 are the kernel variants
enum { CHOICE_COMPACT = mjk::VAR_N };

// kernel variant of the sim's current workspace placement and register budget
int step_variant(const MjmlxBatchedSim* s) {
  if (s->use_gws) return s->high_occ ? mjk::VAR_GWS_OCC : mjk::VAR_GWS;
  if (s->half) return s->high_occ ? mjk::VAR_LDS_OCC_HALF : mjk::VAR_LDS_HALF;
  if (s->high_occ) return mjk::VAR_LDS_OCC;
  return s->big_regs ? mjk::VAR_LDS_BIG : mjk::VAR_LDS;
}

// whether the model needs the kernels for any size: more dofs than the small
// ones take, or more bodies than lanes (LevelBodies)
bool big_kernels(const MjmlxBatchedSim* s) { return s->nv > mjk::SPARSE_ROWS_NV || s->nb > 64; }

// step_variant for the launch: small models with elliptic cones have kernels with
// the register routines, except at 168 VGPRs and on 32 lanes
int launch_variant(const MjmlxBatchedSim* s) {
  int v = step_variant(s);
  bool regs = v == mjk::VAR_LDS || v == mjk::VAR_GWS || v == mjk::VAR_LDS_BIG;
  return regs && !big_kernels(s) && s->model.cone != mjh::CONE_PYRAMIDAL ? v | mjk::VAR_CONES : v;
}

// one workgroup (one wave) per env: the kernel variant for the workspace
// placement (device memory, LDS at three, two or one waves per SIMD), compiled
// for the model's narrow-phase set and, with sensors, the sensor stage
void launch_step(MjmlxBatchedSim* s, mjk::StepIO io, int nsub) {
  if (s->compact && nsub > 0 && !io.dump1 && !io.dump2) {
    size_t bytes = s->Lc.total * sizeof(float);
    io.redo = s->d_redo;
    io.redo_pass = 1;
    mjk::StepLaunch c{s->d_kpc, s->B, 0, s->compact_variant, bytes, nullptr, s->stream, 0};
    mjk::launch_step_np(s->npset, true, c, io, nsub);
    io.redo_pass = 2;
  }
  mjk::StepLaunch l{s->d_kp, s->B, 0, launch_variant(s), s->lds_bytes, s->d_gws, s->stream,
                    mjk::ls_cache_rows(s->L.maxefc)};
  mjk::launch_step_np(s->npset | (s->model.nsensor > 0 ? 4 : 0), big_kernels(s), l, io, nsub);
}

mjk::StepIO make_io(MjmlxBatchedSim* s, float* dump1, float* dump2) {
  mjk::StepIO io{};
  io.qpos = s->d_qpos; io.qvel = s->d_qvel; io.qacc_ws = s->d_qws; io.ctrl = s->d_ctrl;
  io.niter = s->d_niter; io.status = s->d_status; io.ncon = s->d_ncon; io.nefc = s->d_nefc;
  io.dump1 = dump1; io.dump2 = dump2;
  io.has_aux = s->aux_on ? 1 : 0;
  io.aux.xpos = s->d_aux[0]; io.aux.xquat = s->d_aux[1]; io.aux.subtree_com = s->d_aux[2];
  io.aux.cinert = s->d_aux[3]; io.aux.cvel = s->d_aux[4]; io.aux.qfrc_actuator = s->d_aux[5];
  io.aux.cfrc_ext = s->d_aux[6];
  io.rand = s->d_rand; io.nrand = s->nrand;
  io.sensordata = s->d_sensordata; io.sens_prev = s->d_sens_prev;
  io.order = s->d_ident;
  return io;
}

void upload_ctrl(MjmlxBatchedSim* s, const float* ctrl) {
  size_t n = (size_t)s->B * std::max(s->nu, 1);
  if (ctrl && s->nu > 0) {
    // the previous upload must have left the pinned staging buffer before it is rewritten
    if (s->ctrl_pending) HIPOK(hipEventSynchronize(s->ev_ctrl));
    std::memcpy(s->h_ctrl, ctrl, (size_t)s->B * s->nu * sizeof(float));
    HIPOK(hipMemcpyAsync(s->d_ctrl, s->h_ctrl, (size_t)s->B * s->nu * sizeof(float), hipMemcpyHostToDevice, s->stream));
    HIPOK(hipEventRecord(s->ev_ctrl, s->stream));
    s->ctrl_pending = true;
  } else if (s->nu > 0 && !s->ctrl_zero) {
    // no ctrl: zero it once; later NULL calls find it zero already
    HIPOK(hipMemsetAsync(s->d_ctrl, 0, n * sizeof(float), s->stream));
  }
  s->ctrl_zero = !(ctrl && s->nu > 0);
}

void launch(MjmlxBatchedSim* s, int nsub, float* dump1, float* dump2) {
  mjk::StepIO io = make_io(s, dump1, dump2);
  HIPOK(hipEventRecord(s->ev0, s->stream));
  bool order = s->order_mode >= 0 ? s->order_mode == 1 : s->B >= 16 * std::max(1, s->ncu);
  if (order && nsub > 0 && s->B > 1) {
    hipLaunchKernelGGL(k_order, dim3(1), dim3(1024), 0, s->stream, s->d_niter, s->d_order, s->B);
    io.order = s->d_order;
  }
  launch_step(s, io, nsub);
  HIPOK(hipGetLastError());
  HIPOK(hipEventRecord(s->ev1, s->stream));
  s->timed = true;
}

void ensure_learned(MjmlxBatchedSim* s) {
  if (s->d_pred) return;
  size_t nf = (size_t)s->B * (s->dm.nfeat + s->nv);
  for (int i = 0; i < 2; i++) {
    HIPOK(hipMalloc(&s->d_feat[i], nf * sizeof(float)));
    HIPOK(hipMemsetAsync(s->d_feat[i], 0, nf * sizeof(float), s->stream));
  }
  HIPOK(hipMalloc(&s->d_pred, (size_t)s->B * std::max(1, s->nv) * sizeof(float)));
  HIPOK(hipMemsetAsync(s->d_pred, 0, (size_t)s->B * std::max(1, s->nv) * sizeof(float), s->stream));
  s->feat_valid = false;
}

// One launch per substep. With warm-start mode 2 the network predicts each
// substep's qacc from the previous substep's features and this call's ctrl
// before the launch; with `rec` every substep that has input features appends
// (features, converged qacc) rows to rec's training set.
// The learned control step's launches (features, network, one step launch per
// substep), issued on the sim's stream; feat_cur alternates per substep.
void issue_learned(MjmlxBatchedSim* s, int n, int cur) {
  int coff = s->nq + s->nv;
  for (int k = 0; k < n; k++) {
    mjk::StepIO io = make_io(s, nullptr, nullptr);
    io.accumulate = k > 0;
    int nf = s->nfeat();
    const float* base = s->feat_mode ? s->d_feat[cur] + s->dm.nfeat : nullptr;
    mjmlp::predict(s->mlp, s->d_feat[cur], s->d_ctrl, coff, s->nu, s->B, s->d_pred, s->stream, base, nf);
    io.qacc_pred = s->d_pred;
    io.feat = s->d_feat[cur ^ 1];
    io.feat_prev_qacc = s->feat_mode;
    launch_step(s, io, 1);
    cur ^= 1;
  }
}

// Replays the learned control step as a HIP graph, captured again whenever
// what its launches bake in changes (substep count, feature buffer parity,
// network and its buffers, feature mode, kernel variant). Returns false when
// the graph path does not apply (no network or no features yet).
bool step_graph(MjmlxBatchedSim* s, int n) {
  if (!s->graph_on || s->ws_mode != 2 || !s->mlp || !s->feat_valid) return false;
  s->mlp->ensure(s->B);  // allocations happen before any capture
  if (!s->gexec || s->g_n != n || s->g_cur != s->feat_cur || s->g_mlp != s->mlp || s->g_xb != s->mlp->xb ||
      s->g_mode != s->feat_mode || s->g_gws != s->use_gws || s->g_occ != s->high_occ || s->g_big != s->big_regs ||
      s->g_half != s->half || s->g_compact != s->compact) {
    if (s->gexec) { HIPOK(hipGraphExecDestroy(s->gexec)); s->gexec = nullptr; }
    if (s->graph) { HIPOK(hipGraphDestroy(s->graph)); s->graph = nullptr; }
    HIPOK(hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal));
    issue_learned(s, n, s->feat_cur);
    HIPOK(hipStreamEndCapture(s->stream, &s->graph));
    HIPOK(hipGraphInstantiate(&s->gexec, s->graph, nullptr, nullptr, 0));
    s->g_n = n; s->g_cur = s->feat_cur; s->g_mlp = s->mlp; s->g_xb = s->mlp->xb;
    s->g_mode = s->feat_mode; s->g_gws = s->use_gws; s->g_occ = s->high_occ; s->g_big = s->big_regs;
    s->g_half = s->half; s->g_compact = s->compact;
  }
  HIPOK(hipEventRecord(s->ev0, s->stream));
  HIPOK(hipGraphLaunch(s->gexec, s->stream));
  HIPOK(hipEventRecord(s->ev1, s->stream));
  s->timed = true;
  s->feat_cur ^= n & 1;
  return true;
}

long step_substeps(MjmlxBatchedSim* s, int n, MjmlxMLP* rec) {
  ensure_learned(s);
  if (!rec && step_graph(s, n)) return 0;
  long rows = 0;
  int coff = s->nq + s->nv;
  HIPOK(hipEventRecord(s->ev0, s->stream));
  for (int k = 0; k < n; k++) {
    mjk::StepIO io = make_io(s, nullptr, nullptr);
    io.accumulate = k > 0;
    int nf = s->nfeat();
    const float* base = s->feat_mode ? s->d_feat[s->feat_cur] + s->dm.nfeat : nullptr;
    if (s->ws_mode == 2 && s->mlp && s->feat_valid) {
      mjmlp::predict(s->mlp, s->d_feat[s->feat_cur], s->d_ctrl, coff, s->nu, s->B, s->d_pred, s->stream, base, nf);
      io.qacc_pred = s->d_pred;
    }
    io.feat = s->d_feat[s->feat_cur ^ 1];
    io.feat_prev_qacc = s->feat_mode;
    launch_step(s, io, 1);
    HIPOK(hipGetLastError());
    if (rec && s->feat_valid)
      rows += mjmlp::record(rec, s->d_feat[s->feat_cur], s->d_ctrl, coff, s->nu, s->d_qws, s->B, s->stream, base, nf);
    s->feat_cur ^= 1;
    s->feat_valid = true;
  }
  HIPOK(hipEventRecord(s->ev1, s->stream));
  s->timed = true;
  return rows;
}

// Warm-start mode 3: one network pass per call on the features the previous
// call left (the state this call starts from) and one fused launch of all
// substeps, whose first substep takes the prediction as a candidate.
void step_first_learned(MjmlxBatchedSim* s, int n) {
  ensure_learned(s);
  mjk::StepIO io = make_io(s, nullptr, nullptr);
  HIPOK(hipEventRecord(s->ev0, s->stream));
  if (s->mlp && s->feat_valid) {
    const float* base = s->feat_mode ? s->d_feat[s->feat_cur] + s->dm.nfeat : nullptr;
    mjmlp::predict(s->mlp, s->d_feat[s->feat_cur], s->d_ctrl, s->nq + s->nv, s->nu, s->B, s->d_pred, s->stream, base,
                   s->nfeat());
    io.qacc_pred = s->d_pred;
  }
  io.feat = s->d_feat[s->feat_cur ^ 1];
  io.feat_prev_qacc = s->feat_mode;
  launch_step(s, io, n);
  HIPOK(hipGetLastError());
  HIPOK(hipEventRecord(s->ev1, s->stream));
  s->timed = true;
  s->feat_cur ^= 1;
  s->feat_valid = true;
}

void ensure_aux(MjmlxBatchedSim* s) {
  if (s->aux_on) return;
  for (int i = 0; i < 7; i++) {
    size_t n = std::max<size_t>(1, s->aux_len(i));
    HIPOK(hipMalloc(&s->d_aux[i], n * sizeof(float)));
    HIPOK(hipMemsetAsync(s->d_aux[i], 0, n * sizeof(float), s->stream));
    HIPOK(hipHostMalloc(&s->h_aux[i], n * sizeof(float), hipHostMallocDefault));
  }
  s->aux_on = true;
  // derived quantities of the current state (no integration)
  launch(s, 0, nullptr, nullptr);
}

const float* get_aux(const MjmlxBatchedSim* cs, int i, int* n_out) {
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  if (!s) return nullptr;
  try {
    ensure_aux(s);
    size_t n = s->aux_len(i);
    HIPOK(hipMemcpyAsync(s->h_aux[i], s->d_aux[i], n * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    if (n_out) *n_out = (int)n;
    return s->h_aux[i];
  } catch (const std::exception& e) {
    report("mjmlx_batched_get_*", e);
    return nullptr;
  }
}

std::string read_file(const char* path) {
  std::ifstream f(path, std::ios::binary);
  if (!f) throw std::runtime_error(std::string("cannot open ") + path);
  std::stringstream ss;
  ss << f.rdbuf();
  return ss.str();
}

MjmlxModel* load(const std::string& xml, const MjmlxModelOptions* o, const char* fn) {
  try {
    auto* h = new MjmlxModel();
    if (o) { h->opt.self_collision = o->self_collision; h->opt.max_condim = o->max_condim; }
    h->m = mjh::compile_mjcf(xml, h->opt);
    return h;
  } catch (const std::exception& e) {
    report(fn, e);
    return nullptr;
  }
}

void removed(const char* fn) {
  std::fprintf(stderr, "%s error: the single-env pipeline is not available; use the batched API\n", fn);
}

}  // namespace

// ------------------------------------------------------------------ C API
extern "C" {

MJMLX_API const char* mjmlx_version(void) { return "mjmlx-hip 0.1.0 (gfx950)"; }

MJMLX_API int mjmlx_hip_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

MJMLX_API MjmlxModel* mjmlx_load_model(const char* xml_path) {
  if (!xml_path) return nullptr;
  try { return load(read_file(xml_path), nullptr, "mjmlx_load_model"); }
  catch (const std::exception& e) { report("mjmlx_load_model", e); return nullptr; }
}
MJMLX_API MjmlxModel* mjmlx_load_model_from_string(const char* xml) {
  if (!xml) return nullptr;
  return load(xml, nullptr, "mjmlx_load_model_from_string");
}
MJMLX_API MjmlxModelOptions mjmlx_default_model_options(void) {
  MjmlxModelOptions o;
  o.self_collision = 1;
  o.max_condim = 0;
  return o;
}
MJMLX_API MjmlxModel* mjmlx_load_model_ex(const char* xml_path, const MjmlxModelOptions* options) {
  if (!xml_path) return nullptr;
  try { return load(read_file(xml_path), options, "mjmlx_load_model_ex"); }
  catch (const std::exception& e) { report("mjmlx_load_model_ex", e); return nullptr; }
}
MJMLX_API MjmlxModel* mjmlx_load_model_from_string_ex(const char* xml, const MjmlxModelOptions* options) {
  if (!xml) return nullptr;
  return load(xml, options, "mjmlx_load_model_from_string_ex");
}
MJMLX_API void mjmlx_free_model(MjmlxModel* model) { delete model; }

MJMLX_API MjmlxModelInfo mjmlx_model_info(const MjmlxModel* model) {
  MjmlxModelInfo i;
  std::memset(&i, 0, sizeof(i));
  if (!model) return i;
  const auto& m = model->m;
  i.nq = m.nq; i.nv = m.nv; i.nu = m.nu; i.na = 0; i.nbody = m.nbody; i.njnt = m.njnt; i.ngeom = m.ngeom;
  i.nsite = m.nsite;
  try { i.ncon = mjh::max_contacts(m, mjh::build_pairs(m)); } catch (...) { i.ncon = 0; }
  return i;
}

MJMLX_API float mjmlx_model_opt_timestep(const MjmlxModel* model) { return model ? (float)model->m.timestep : 0.f; }
MJMLX_API void mjmlx_model_set_opt_timestep(MjmlxModel* model, float dt) { if (model && dt > 0) model->m.timestep = dt; }
MJMLX_API float mjmlx_model_body_mass(const MjmlxModel* model, int body_id) {
  if (!model || body_id < 0 || body_id >= model->m.nbody) return 0.f;
  return (float)model->m.body_mass[body_id];
}
MJMLX_API int mjmlx_name2id(const MjmlxModel* model, int obj_type, const char* name) {
  if (!model || !name) return -1;
  return model->m.name2id(obj_type, name);
}
MJMLX_API const char* mjmlx_id2name(const MjmlxModel* model, int obj_type, int id) {
  return model ? model->m.id2name(obj_type, id) : nullptr;
}
// sensors of the compiled model (reference src/sensor.cpp:362-377)
MJMLX_API int mjmlx_model_nsensor(const MjmlxModel* model) { return model ? model->m.nsensor : 0; }
MJMLX_API int mjmlx_model_nsensordata(const MjmlxModel* model) { return model ? model->m.nsensordata : 0; }
MJMLX_API const char* mjmlx_model_sensor_name(const MjmlxModel* model, int i) {
  if (!model || i < 0 || i >= model->m.nsensor) return nullptr;
  return model->m.sensor_name[i].c_str();
}
MJMLX_API int mjmlx_model_sensor_type(const MjmlxModel* model, int i) {
  return model && i >= 0 && i < model->m.nsensor ? model->m.sensor_type[i] : -1;
}
MJMLX_API int mjmlx_model_sensor_adr(const MjmlxModel* model, int i) {
  return model && i >= 0 && i < model->m.nsensor ? model->m.sensor_adr[i] : -1;
}
MJMLX_API int mjmlx_model_sensor_dim(const MjmlxModel* model, int i) {
  return model && i >= 0 && i < model->m.nsensor ? model->m.sensor_dim[i] : -1;
}
MJMLX_API const void* mjmlx_get_mj_model(const MjmlxModel*) { return nullptr; }

MJMLX_API int mjmlx_model_field(const MjmlxModel* model, const char* name, double* out, int cap) {
  if (!model || !name) return -1;
  try { return mjh::model_field(model->m, name, out, cap); }
  catch (const std::exception& e) { report("mjmlx_model_field", e); return -1; }
}

// ---- single-env (removed)
MJMLX_API MjmlxData* mjmlx_make_data(const MjmlxModel*) { removed("mjmlx_make_data"); return nullptr; }
MJMLX_API void mjmlx_free_data(MjmlxData* data) { delete data; }
MJMLX_API void mjmlx_reset_data(const MjmlxModel*, MjmlxData*) { removed("mjmlx_reset_data"); }
MJMLX_API void mjmlx_forward(const MjmlxModel*, MjmlxData*) { removed("mjmlx_forward"); }
MJMLX_API void mjmlx_step(const MjmlxModel*, MjmlxData*) { removed("mjmlx_step"); }
MJMLX_API void mjmlx_step1(const MjmlxModel*, MjmlxData*) { removed("mjmlx_step1"); }
MJMLX_API void mjmlx_step2(const MjmlxModel*, MjmlxData*) { removed("mjmlx_step2"); }
MJMLX_API void mjmlx_kinematics(const MjmlxModel*, MjmlxData*) { removed("mjmlx_kinematics"); }
MJMLX_API void mjmlx_set_qpos(MjmlxData*, const float*, int) { removed("mjmlx_set_qpos"); }
MJMLX_API void mjmlx_set_qvel(MjmlxData*, const float*, int) { removed("mjmlx_set_qvel"); }
MJMLX_API void mjmlx_set_ctrl(MjmlxData*, const float*, int) { removed("mjmlx_set_ctrl"); }
#define MJMLX_SINGLE_GETTER(fn)                                  \
  MJMLX_API const float* fn(const MjmlxData*, int* n_out) {      \
    if (n_out) *n_out = 0;                                       \
    removed(#fn);                                                \
    return nullptr;                                              \
  }
MJMLX_SINGLE_GETTER(mjmlx_get_qpos)
MJMLX_SINGLE_GETTER(mjmlx_get_qvel)
MJMLX_SINGLE_GETTER(mjmlx_get_ctrl)
MJMLX_SINGLE_GETTER(mjmlx_get_xpos)
MJMLX_SINGLE_GETTER(mjmlx_get_xquat)
MJMLX_SINGLE_GETTER(mjmlx_get_xipos)
MJMLX_SINGLE_GETTER(mjmlx_get_cvel)
MJMLX_SINGLE_GETTER(mjmlx_get_qfrc_bias)
MJMLX_SINGLE_GETTER(mjmlx_get_qacc)
MJMLX_SINGLE_GETTER(mjmlx_get_qfrc_constraint)
MJMLX_SINGLE_GETTER(mjmlx_get_qfrc_actuator)
MJMLX_SINGLE_GETTER(mjmlx_get_qfrc_passive)
MJMLX_SINGLE_GETTER(mjmlx_get_qfrc_gravcomp)
MJMLX_SINGLE_GETTER(mjmlx_get_qfrc_smooth)
MJMLX_SINGLE_GETTER(mjmlx_get_qacc_smooth)
MJMLX_SINGLE_GETTER(mjmlx_get_subtree_com)
MJMLX_SINGLE_GETTER(mjmlx_get_cinert)
MJMLX_SINGLE_GETTER(mjmlx_get_cfrc_ext)
#undef MJMLX_SINGLE_GETTER
MJMLX_API int mjmlx_get_ncon(const MjmlxData*) { return 0; }
MJMLX_API int mjmlx_get_nefc(const MjmlxData*) { return 0; }
MJMLX_API void mjmlx_rne_post_constraint(const MjmlxModel*, MjmlxData*) { removed("mjmlx_rne_post_constraint"); }

// ---- batched
MJMLX_API MjmlxBatchedSim* mjmlx_batched_create(const MjmlxModel* model, const MjmlxBatchedConfig* config) {
  if (!model || !config) return nullptr;
  MjmlxBatchedSim* s = nullptr;
  try {
    if (config->num_envs <= 0) throw std::runtime_error("num_envs must be positive");
    if (!config->use_gpu)
      throw std::runtime_error("use_gpu=0 requests the MuJoCo C CPU path, which is not part of the HIP engine");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) throw std::runtime_error("no HIP device available");
    s = new MjmlxBatchedSim();
    s->model = model->m;
    auto& m = s->model;
    if (config->solver_iterations > 0) m.iterations = config->solver_iterations;
    switch (config->integrator) {
      case MJMLX_INTEGRATOR_EULER: m.integrator = mjh::INT_EULER; break;
      case MJMLX_INTEGRATOR_IMPLICIT: m.integrator = mjh::INT_IMPLICIT; break;
      case MJMLX_INTEGRATOR_IMPLICITFAST: m.integrator = mjh::INT_IMPLICITFAST; break;
      default: throw std::runtime_error("the RK4 integrator is not implemented by the HIP engine");
    }
    std::vector<mjh::CollisionPair> pairs;
    s->blob = mjh::build_blob(m, &pairs);
    for (auto& p : pairs) {
      int t1 = m.geom_type[p.g1], t2 = m.geom_type[p.g2];
      if ((t1 == mjk::GCAPSULE && t2 == mjk::GBOX) || (t1 == mjk::GBOX && t2 == mjk::GBOX)) s->npset = std::max(s->npset, 1);
      if (t1 == mjk::GELLIPSOID || t1 == mjk::GCYLINDER || t2 == mjk::GELLIPSOID || t2 == mjk::GCYLINDER) s->npset = 2;
    }
    s->B = config->num_envs; s->nq = m.nq; s->nv = m.nv; s->nu = m.nu; s->nb = m.nbody;
    // per-env capacities: the reference's contact cap and row budget
    int con_over = 0, efc_over = 0;
    if (const char* v = std::getenv("MJMLX_HIP_MAXCON")) con_over = std::max(1, std::atoi(v));
    if (const char* v = std::getenv("MJMLX_HIP_MAXEFC")) efc_over = std::max(1, std::atoi(v));
    mjh::Caps caps = mjh::default_caps(m, pairs, con_over, efc_over);
    // domain randomisation (reference src/batched.cpp:1348-1361): each env's
    // parameter block rides in its workspace
    for (int j = 0; j < m.njnt; j++) s->nfree += m.jnt_type[j] == mjk::JFREE;
    if (config->domain_rand) s->nrand = mjk::rand_size(m.nbody, m.nu, s->nfree);
    s->L = mjk::make_layout(m.nq, m.nv, m.nu, m.nbody, m.njnt, m.ngeom, caps.maxcon, caps.maxefc,
                            m.solver == mjh::SOL_NEWTON, s->nrand, s->blob.proto.jw, s->blob.proto.nM);
    s->L.efc_cap = caps.efc_cap;
    s->L.con_cap = caps.con_cap;
    s->fields = mjh::layout_fields(m, s->L);
    s->lds_bytes = (size_t)s->L.total * sizeof(float);
    int dev = 0;
    HIPOK(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    HIPOK(hipGetDeviceProperties(&prop, dev));
    s->ncu = prop.multiProcessorCount;
    // workspaces beyond lds_max (144 KB unless MJMLX_HIP_LDS_MAX says
    // otherwise, at most the workgroup's LDS) live in device memory instead of
    // LDS. Measured on the box workloads: one LDS-resident env per CU still
    // beats device memory up to ~140 KB workspaces, not at ~158 KB.
    size_t lds_max = 147456;
    if (const char* v = std::getenv("MJMLX_HIP_LDS_MAX")) lds_max = (size_t)std::max(0L, std::atol(v));
    bool use_gws = s->lds_bytes > lds_max || s->lds_bytes > (size_t)prop.sharedMemPerBlock;
    if (const char* v = std::getenv("MJMLX_HIP_GLOBAL_WORKSPACE")) use_gws = use_gws || std::atoi(v) != 0;
    s->lds_ok = s->lds_bytes <= (size_t)prop.sharedMemPerBlock;
    s->use_gws = use_gws;
    size_t lds_cu = prop.maxSharedMemoryPerMultiProcessor > 0 ? (size_t)prop.maxSharedMemoryPerMultiProcessor : 163840;
    s->high_occ = !use_gws && lds_cu / std::max<size_t>(s->lds_bytes, 1) > 8;
    if (const char* v = std::getenv("MJMLX_HIP_HIGH_OCC")) s->high_occ = std::atoi(v) != 0;
    s->big_regs = !use_gws && !s->high_occ && lds_cu / std::max<size_t>(s->lds_bytes, 1) <= 4;
    if (const char* v = std::getenv("MJMLX_HIP_BIG_REGS")) s->big_regs = !use_gws && !s->high_occ && std::atoi(v) != 0;
    // 32 lanes per env (two envs' workspaces per workgroup) by default for
    // models of at most 8 dofs, at 256 registers: measured faster than every
    // 64-lane variant on hinge chains of 2-8 dofs, slower from 16 dofs on
    // (quadruped 0.6x, humanoid 0.45x: half the waves per CU at the same LDS
    // occupancy), and with more bodies than lanes (two chains of 24 bodies, 8
    // dofs, 64 envs: 0.39 ms per control step, on 64 lanes 0.23).
    // MJMLX_HIP_LANES=32 or 64 forces either; the autotuner times both.
    s->half_ok = s->nv <= mjk::SPARSE_ROWS_NV && 2 * s->lds_bytes <= (size_t)prop.sharedMemPerBlock &&
                 2 * s->lds_bytes <= lds_max;
    s->half = !use_gws && s->half_ok && s->nv <= 8 && s->nb <= 32;
    if (const char* v = std::getenv("MJMLX_HIP_LANES")) s->half = !use_gws && s->half_ok && std::atoi(v) == 32;
    if (s->half) {
      s->big_regs = false;
      s->high_occ = false;
      if (const char* v = std::getenv("MJMLX_HIP_HIGH_OCC")) s->high_occ = std::atoi(v) != 0;
    }
    place_big(s, caps, pairs, lds_cu, lds_max);
    if (s->use_gws && !s->d_gws) HIPOK(hipMalloc(&s->d_gws, (size_t)s->B * s->L.total * sizeof(float)));
    HIPOK(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
    HIPOK(hipEventCreate(&s->ev0));
    HIPOK(hipEventCreate(&s->ev1));
    HIPOK(hipEventCreateWithFlags(&s->ev_ctrl, hipEventDisableTiming));
    HIPOK(hipMalloc(&s->d_blob, s->blob.bytes.size()));
    HIPOK(hipMemcpy(s->d_blob, s->blob.bytes.data(), s->blob.bytes.size(), hipMemcpyHostToDevice));
    s->dm = s->blob.bind(s->d_blob);
    HIPOK(hipMalloc(&s->d_kp, sizeof(mjk::KParams)));
    upload_kparams(s);
    size_t B = s->B;
    HIPOK(hipMalloc(&s->d_qpos, B * std::max(1, m.nq) * sizeof(float)));
    HIPOK(hipMalloc(&s->d_qvel, B * std::max(1, m.nv) * sizeof(float)));
    HIPOK(hipMalloc(&s->d_qws, B * std::max(1, m.nv) * sizeof(float)));
    HIPOK(hipMalloc(&s->d_ctrl, B * std::max(1, m.nu) * sizeof(float)));
    HIPOK(hipMalloc(&s->d_qpos0, std::max(1, m.nq) * sizeof(float)));
    HIPOK(hipMalloc(&s->d_niter, B * sizeof(int)));
    HIPOK(hipMalloc(&s->d_status, B * sizeof(int)));
    HIPOK(hipMalloc(&s->d_ncon, B * sizeof(int)));
    HIPOK(hipMalloc(&s->d_nefc, B * sizeof(int)));
    HIPOK(hipMalloc(&s->d_queue, sizeof(int)));
    HIPOK(hipMalloc(&s->d_order, B * sizeof(int)));
    HIPOK(hipMalloc(&s->d_ident, B * sizeof(int)));
    {
      std::vector<int> iota(B);
      for (size_t e = 0; e < B; e++) iota[e] = (int)e;
      HIPOK(hipMemcpy(s->d_ident, iota.data(), B * sizeof(int), hipMemcpyHostToDevice));
    }
    if (const char* v = std::getenv("MJMLX_HIP_ORDER")) s->order_mode = std::atoi(v) != 0;
    HIPOK(hipMalloc(&s->d_mask, B * sizeof(int)));
    HIPOK(hipHostMalloc(&s->h_qpos, B * std::max(1, m.nq) * sizeof(float), hipHostMallocDefault));
    HIPOK(hipHostMalloc(&s->h_qvel, B * std::max(1, m.nv) * sizeof(float), hipHostMallocDefault));
    HIPOK(hipHostMalloc(&s->h_ctrl, B * std::max(1, m.nu) * sizeof(float), hipHostMallocDefault));
    HIPOK(hipHostMalloc(&s->h_mask, B * sizeof(int), hipHostMallocDefault));
    std::vector<float> q0(m.qpos0.begin(), m.qpos0.end());
    for (size_t e = 0; e < B; e++) std::memcpy(s->h_qpos + e * m.nq, q0.data(), m.nq * sizeof(float));
    HIPOK(hipMemcpy(s->d_qpos, s->h_qpos, B * m.nq * sizeof(float), hipMemcpyHostToDevice));
    HIPOK(hipMemcpy(s->d_qpos0, q0.data(), std::max(1, m.nq) * sizeof(float), hipMemcpyHostToDevice));
    HIPOK(hipMemset(s->d_qvel, 0, B * std::max(1, m.nv) * sizeof(float)));
    HIPOK(hipMemset(s->d_qws, 0, B * std::max(1, m.nv) * sizeof(float)));
    HIPOK(hipMemset(s->d_ctrl, 0, B * std::max(1, m.nu) * sizeof(float)));
    HIPOK(hipMemset(s->d_niter, 0, B * sizeof(int)));
    HIPOK(hipMemset(s->d_status, 0, B * sizeof(int)));
    HIPOK(hipMemset(s->d_ncon, 0, B * sizeof(int)));
    HIPOK(hipMemset(s->d_nefc, 0, B * sizeof(int)));
    if (m.nsensor > 0) {
      size_t nsd = (size_t)m.nsensordata, pst = (size_t)s->dm.nsens_acc * 3 + 1;
      HIPOK(hipMalloc(&s->d_sensordata, B * nsd * sizeof(float)));
      HIPOK(hipHostMalloc(&s->h_sensordata, B * nsd * sizeof(float), hipHostMallocDefault));
      HIPOK(hipMalloc(&s->d_sens_prev, B * pst * sizeof(float)));
      HIPOK(hipMemset(s->d_sensordata, 0, B * nsd * sizeof(float)));
      HIPOK(hipMemset(s->d_sens_prev, 0, B * pst * sizeof(float)));
    }
    if (s->nrand > 0) {
      // identity parameters: unit mass, friction and force scales, no COM shift, no drag
      s->h_rand.assign(B * s->nrand, 0.f);
      for (size_t e = 0; e < B; e++) {
        float* r = s->h_rand.data() + e * s->nrand;
        for (int b = 0; b < m.nbody; b++) r[b] = 1.f;
        r[mjk::rand_fric(m.nbody)] = 1.f;
        for (int u = 0; u < m.nu; u++) r[mjk::rand_gain(m.nbody) + u] = 1.f;
      }
      HIPOK(hipMalloc(&s->d_rand, s->h_rand.size() * sizeof(float)));
      HIPOK(hipMemcpy(s->d_rand, s->h_rand.data(), s->h_rand.size() * sizeof(float), hipMemcpyHostToDevice));
    }
    return s;
  } catch (const std::exception& e) {
    report("mjmlx_batched_create", e);
    free_sim(s);
    return nullptr;
  }
}

MJMLX_API void mjmlx_batched_free(MjmlxBatchedSim* sim) { free_sim(sim); }

MJMLX_API void mjmlx_batched_step_n(MjmlxBatchedSim* sim, const float* ctrl, int n) {
  if (!sim || n <= 0) return;
  try {
    upload_ctrl(sim, ctrl);
    if (sim->ws_mode == 2) step_substeps(sim, n, nullptr);
    else if (sim->ws_mode == 3) step_first_learned(sim, n);
    else launch(sim, n, nullptr, nullptr);
  } catch (const std::exception& e) { report("mjmlx_batched_step_n", e); }
}

MJMLX_API void mjmlx_batched_step(MjmlxBatchedSim* sim, const float* ctrl) { mjmlx_batched_step_n(sim, ctrl, 1); }

// ------------------------------------------------------- allocation-free step
// The per-env workspaces of mjmlx_batched_step_n_noalloc live in this
// file-scope device array (one copy per GPU, held until the process ends)
// instead of memory the library allocates. Host code never uses the array's
// name as an address: each device's address comes from hipGetSymbolAddress,
// taken once per device with that device current.
namespace {
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
constexpr int kMaxDevices = 64;
__device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];
float* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

float* scratch_ptr() {
  int dev = 0;
  HIPOK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("device index beyond the scratch table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    hipError_t rc = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (rc != hipSuccess || !p)
      throw std::runtime_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(rc));
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  return g_scratch_ptr[dev];
}
}  // namespace

MJMLX_API size_t mjmlx_batched_noalloc_scratch_bytes(void) { return kNoAllocScratchBytes; }

MJMLX_API int mjmlx_batched_step_n_noalloc(MjmlxBatchedSim* sim, const float* ctrl, int n) {
  if (!sim || n <= 0) return -1;
  try {
    if (sim->ws_mode == 2 || sim->ws_mode == 3)
      throw std::runtime_error("the learned warm-start modes are not available without allocation");
    size_t need = (size_t)sim->B * sim->L.total * sizeof(float);
    if (need > kNoAllocScratchBytes)
      throw std::runtime_error("the workspaces of " + std::to_string(sim->B) + " envs need " + std::to_string(need) +
                               " bytes, beyond the " + std::to_string(kNoAllocScratchBytes) + "-byte scratch");
    float* ws = scratch_ptr();
    upload_ctrl(sim, ctrl);
    mjk::StepIO io = make_io(sim, nullptr, nullptr);
    int var = sim->use_gws ? step_variant(sim) : mjk::VAR_GWS;
    var |= launch_variant(sim) & mjk::VAR_CONES;  // the arithmetic of the sim's own step
    mjk::StepLaunch l{sim->d_kp, sim->B, 0, var, 0, ws, sim->stream, mjk::ls_cache_rows(sim->L.maxefc)};
    HIPOK(hipEventRecord(sim->ev0, sim->stream));
    mjk::launch_step_np(sim->npset | (sim->model.nsensor > 0 ? 4 : 0), big_kernels(sim), l, io, n);
    HIPOK(hipGetLastError());
    HIPOK(hipEventRecord(sim->ev1, sim->stream));
    sim->timed = true;
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_step_n_noalloc", e); return -1; }
}

MJMLX_API void mjmlx_batched_reset(MjmlxBatchedSim* sim, const int* mask) {
  if (!sim || !mask) return;
  try {
    sim->feat_valid = false;
    std::memcpy(sim->h_mask, mask, sim->B * sizeof(int));
    HIPOK(hipMemcpyAsync(sim->d_mask, sim->h_mask, sim->B * sizeof(int), hipMemcpyHostToDevice, sim->stream));
    hipLaunchKernelGGL(k_reset, dim3((sim->B + 255) / 256), dim3(256), 0, sim->stream, sim->d_mask, sim->d_qpos,
                       sim->d_qvel, sim->d_qws, sim->d_qpos0, sim->B, sim->nq, sim->nv, sim->d_sens_prev,
                       sim->dm.nsens_acc * 3 + 1);
    HIPOK(hipGetLastError());
    HIPOK(hipStreamSynchronize(sim->stream));
  } catch (const std::exception& e) { report("mjmlx_batched_reset", e); }
}

MJMLX_API void mjmlx_batched_get_state(const MjmlxBatchedSim* cs, float* qpos_out, float* qvel_out, int* nq_out, int* nv_out) {
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  if (!s) return;
  try {
    if (nq_out) *nq_out = s->nq;
    if (nv_out) *nv_out = s->nv;
    if (qpos_out) HIPOK(hipMemcpyAsync(s->h_qpos, s->d_qpos, (size_t)s->B * s->nq * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    if (qvel_out) HIPOK(hipMemcpyAsync(s->h_qvel, s->d_qvel, (size_t)s->B * s->nv * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    if (qpos_out) std::memcpy(qpos_out, s->h_qpos, (size_t)s->B * s->nq * sizeof(float));
    if (qvel_out) std::memcpy(qvel_out, s->h_qvel, (size_t)s->B * s->nv * sizeof(float));
  } catch (const std::exception& e) { report("mjmlx_batched_get_state", e); }
}

MJMLX_API void mjmlx_batched_set_state(MjmlxBatchedSim* s, const float* qpos, const float* qvel) {
  if (!s) return;
  try {
    s->feat_valid = false;
    HIPOK(hipStreamSynchronize(s->stream));
    if (qpos) {
      std::memcpy(s->h_qpos, qpos, (size_t)s->B * s->nq * sizeof(float));
      HIPOK(hipMemcpyAsync(s->d_qpos, s->h_qpos, (size_t)s->B * s->nq * sizeof(float), hipMemcpyHostToDevice, s->stream));
    }
    if (qvel) {
      std::memcpy(s->h_qvel, qvel, (size_t)s->B * s->nv * sizeof(float));
      HIPOK(hipMemcpyAsync(s->d_qvel, s->h_qvel, (size_t)s->B * s->nv * sizeof(float), hipMemcpyHostToDevice, s->stream));
    }
    HIPOK(hipStreamSynchronize(s->stream));
  } catch (const std::exception& e) { report("mjmlx_batched_set_state", e); }
}

MJMLX_API const float* mjmlx_batched_get_qpos(const MjmlxBatchedSim* cs, int* n_out) {
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  if (!s) return nullptr;
  try {
    HIPOK(hipMemcpyAsync(s->h_qpos, s->d_qpos, (size_t)s->B * s->nq * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    if (n_out) *n_out = s->B * s->nq;
    return s->h_qpos;
  } catch (const std::exception& e) { report("mjmlx_batched_get_qpos", e); return nullptr; }
}

MJMLX_API const float* mjmlx_batched_get_qvel(const MjmlxBatchedSim* cs, int* n_out) {
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  if (!s) return nullptr;
  try {
    HIPOK(hipMemcpyAsync(s->h_qvel, s->d_qvel, (size_t)s->B * s->nv * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    if (n_out) *n_out = s->B * s->nv;
    return s->h_qvel;
  } catch (const std::exception& e) { report("mjmlx_batched_get_qvel", e); return nullptr; }
}

MJMLX_API const float* mjmlx_batched_get_xpos(const MjmlxBatchedSim* s, int* n) { return get_aux(s, 0, n); }
MJMLX_API const float* mjmlx_batched_get_xquat(const MjmlxBatchedSim* s, int* n) { return get_aux(s, 1, n); }
MJMLX_API const float* mjmlx_batched_get_subtree_com(const MjmlxBatchedSim* s, int* n) { return get_aux(s, 2, n); }
MJMLX_API const float* mjmlx_batched_get_cinert(const MjmlxBatchedSim* s, int* n) { return get_aux(s, 3, n); }
MJMLX_API const float* mjmlx_batched_get_cvel(const MjmlxBatchedSim* s, int* n) { return get_aux(s, 4, n); }
MJMLX_API const float* mjmlx_batched_get_qfrc_actuator(const MjmlxBatchedSim* s, int* n) { return get_aux(s, 5, n); }
MJMLX_API const float* mjmlx_batched_get_cfrc_ext(const MjmlxBatchedSim* s, int* n) { return get_aux(s, 6, n); }
MJMLX_API int mjmlx_batched_nsensordata(const MjmlxBatchedSim* s) { return s ? s->model.nsensordata : 0; }

// Sensor values [num_envs][nsensordata] at the start of the last physics
// substep of the last step (reference src/batched.cpp:1635-1651, sensor.cpp:
// the outputs of a step describe the state it started from); NULL without
// sensors. Valid until the next step, set or free.
MJMLX_API const float* mjmlx_batched_get_sensordata(const MjmlxBatchedSim* cs, int* n_out) {
  if (n_out) *n_out = 0;
  if (!cs || cs->model.nsensordata == 0) return nullptr;
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  try {
    size_t n = (size_t)s->B * s->model.nsensordata;
    HIPOK(hipMemcpyAsync(s->h_sensordata, s->d_sensordata, n * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    if (n_out) *n_out = (int)n;
    return s->h_sensordata;
  } catch (const std::exception& e) { report("mjmlx_batched_get_sensordata", e); return nullptr; }
}

MJMLX_API void mjmlx_batched_set_env_qpos(MjmlxBatchedSim* s, int env, const float* qpos, int nq) {
  if (!s || !qpos || env < 0 || env >= s->B || nq != s->nq) return;
  s->feat_valid = false;
  try {
    HIPOK(hipStreamSynchronize(s->stream));
    HIPOK(hipMemcpy(s->d_qpos + (size_t)env * s->nq, qpos, s->nq * sizeof(float), hipMemcpyHostToDevice));
  } catch (const std::exception& e) { report("mjmlx_batched_set_env_qpos", e); }
}
MJMLX_API void mjmlx_batched_set_env_qvel(MjmlxBatchedSim* s, int env, const float* qvel, int nv) {
  if (!s || !qvel || env < 0 || env >= s->B || nv != s->nv) return;
  s->feat_valid = false;
  try {
    HIPOK(hipStreamSynchronize(s->stream));
    HIPOK(hipMemcpy(s->d_qvel + (size_t)env * s->nv, qvel, s->nv * sizeof(float), hipMemcpyHostToDevice));
  } catch (const std::exception& e) { report("mjmlx_batched_set_env_qvel", e); }
}

namespace {
// uploads the host parameter blocks once the steps queued before have read the old ones
void upload_rand(MjmlxBatchedSim* s) {
  HIPOK(hipStreamSynchronize(s->stream));
  HIPOK(hipMemcpy(s->d_rand, s->h_rand.data(), s->h_rand.size() * sizeof(float), hipMemcpyHostToDevice));
}
}  // namespace

// Per-env physical parameters of a sim created with domain_rand (reference
// src/batched.cpp:1508-1526): rows i of the arrays go to env env_idx[i] (env i
// when env_idx is NULL, then n must be num_envs); NULL arrays are left as
// they are. Returns 0, -1 (bad handle, no domain_rand, bad n), -2 (env index
// out of range).
MJMLX_API int mjmlx_batched_set_env_params(MjmlxBatchedSim* s, const int* env_idx, int n, const float* mass_scale,
                                           const float* com_delta, const float* friction_scale,
                                           const float* gain_scale) {
  if (!s || s->nrand == 0 || n < 0) return -1;
  if (!env_idx && n != s->B) return -1;
  for (int i = 0; i < n; i++)
    if (env_idx && (env_idx[i] < 0 || env_idx[i] >= s->B)) return -2;
  try {
    int nb = s->nb, nu = s->nu;
    for (int i = 0; i < n; i++) {
      float* r = s->h_rand.data() + (size_t)(env_idx ? env_idx[i] : i) * s->nrand;
      if (mass_scale) std::memcpy(r, mass_scale + (size_t)i * nb, nb * sizeof(float));
      if (com_delta) std::memcpy(r + mjk::rand_com(nb), com_delta + (size_t)i * nb * 3, nb * 3 * sizeof(float));
      if (friction_scale) r[mjk::rand_fric(nb)] = friction_scale[i];
      if (gain_scale && nu > 0) std::memcpy(r + mjk::rand_gain(nb), gain_scale + (size_t)i * nu, nu * sizeof(float));
    }
    upload_rand(s);
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_set_env_params", e); return -1; }
}

// Quadratic drag coefficient k of each free joint (F = -k |v| v), drag_k
// [n][num_free_joints] (reference src/batched.cpp:1528-1541). Returns 0, -1
// (bad handle / arguments, no domain_rand), -2 (env index out of range), -3
// (the model has no free joint).
MJMLX_API int mjmlx_batched_set_free_drag(MjmlxBatchedSim* s, const int* env_idx, int n, const float* drag_k) {
  if (!s || s->nrand == 0 || n < 0 || !drag_k) return -1;
  if (s->nfree == 0) return -3;
  if (!env_idx && n != s->B) return -1;
  for (int i = 0; i < n; i++)
    if (env_idx && (env_idx[i] < 0 || env_idx[i] >= s->B)) return -2;
  try {
    for (int i = 0; i < n; i++) {
      float* r = s->h_rand.data() + (size_t)(env_idx ? env_idx[i] : i) * s->nrand;
      std::memcpy(r + mjk::rand_drag(s->nb, s->nu), drag_k + (size_t)i * s->nfree, s->nfree * sizeof(float));
    }
    upload_rand(s);
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_set_free_drag", e); return -1; }
}

// free joints of the model when the sim has domain_rand, else 0 (reference src/batched.cpp:1543-1545)
MJMLX_API int mjmlx_batched_num_free_joints(const MjmlxBatchedSim* s) { return s && s->nrand > 0 ? s->nfree : 0; }

MJMLX_API int mjmlx_batched_set_pack_spec(MjmlxBatchedSim* s, const int* body_ids, int nsel, int dof_lo, int ndof) {
  if (!s || nsel < 0 || ndof < 0 || (nsel > 0 && !body_ids)) return -1;
  for (int i = 0; i < nsel; i++) if (body_ids[i] < 0 || body_ids[i] >= s->nb) return -1;
  if (dof_lo < 0 || dof_lo + ndof > s->nv) return -1;
  try {
    if (s->d_pack_bodies) { hipFree(s->d_pack_bodies); s->d_pack_bodies = nullptr; }
    if (s->d_pack) { hipFree(s->d_pack); s->d_pack = nullptr; }
    HIPOK(hipMalloc(&s->d_pack_bodies, std::max(1, nsel) * sizeof(int)));
    if (nsel > 0) HIPOK(hipMemcpy(s->d_pack_bodies, body_ids, nsel * sizeof(int), hipMemcpyHostToDevice));
    s->pack_stride = s->nq + s->nv + nsel + 2;
    HIPOK(hipMalloc(&s->d_pack, (size_t)s->B * s->pack_stride * sizeof(float)));
    s->pack_nsel = nsel; s->pack_lo = dof_lo; s->pack_ndof = ndof;
    ensure_aux(s);
    return s->pack_stride;
  } catch (const std::exception& e) { report("mjmlx_batched_set_pack_spec", e); return -1; }
}

MJMLX_API int mjmlx_batched_get_pack(MjmlxBatchedSim* s, float* out) {
  if (!s || !out || s->pack_stride < 0) return -1;
  try {
    hipLaunchKernelGGL(k_pack, dim3((s->B + 127) / 128), dim3(128), 0, s->stream, s->d_qpos, s->d_qvel, s->d_aux[6],
                       s->d_aux[5], s->d_pack_bodies, s->pack_nsel, s->pack_lo, s->pack_ndof, s->B, s->nq, s->nv, s->nb,
                       s->d_pack);
    HIPOK(hipGetLastError());
    HIPOK(hipMemcpyAsync(out, s->d_pack, (size_t)s->B * s->pack_stride * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_get_pack", e); return -1; }
}

// mj_ray from pnt along vec ([num_envs][nray][3] each) against each env's
// geoms at its current qpos: dist in units of |vec| and the geom id, or -1 /
// -1. Geoms of body bodyexclude, of groups switched off in geomgroup[6] (NULL:
// all groups) and, when flg_static is 0, of bodies welded to the world are
// skipped. Returns 0, or -1 (bad arguments). Reference
// src/batched.cpp:1846-1893.
MJMLX_API int mjmlx_batched_raycast(MjmlxBatchedSim* s, const float* pnt, const float* vec, int nray, int bodyexclude,
                                   const unsigned char* geomgroup, int flg_static, float* dist_out, int* geomid_out) {
  if (!s || !pnt || !vec || !dist_out || !geomid_out || nray <= 0) return -1;
  try {
    const auto& m = s->model;
    size_t total = (size_t)s->B * nray;
    if (m.ngeom == 0) {
      std::fill(dist_out, dist_out + total, -1.f);
      std::fill(geomid_out, geomid_out + total, -1);
      return 0;
    }
    std::vector<int> mask(m.ngeom);
    for (int g = 0; g < m.ngeom; g++) {
      int b = m.geom_bodyid[g], grp = m.geom_group[g];
      bool group_ok = !geomgroup || (grp >= 0 && grp < 6 && geomgroup[grp]);
      bool static_ok = flg_static || m.body_weldid[b] != 0;
      mask[g] = b != bodyexclude && group_ok && static_ok;
    }
    if (total > s->ray_cap) {
      for (void* p : {(void*)s->d_rays, (void*)s->d_rdist, (void*)s->d_rgid}) if (p) HIPOK(hipFree(p));
      s->d_rays = nullptr; s->d_rdist = nullptr; s->d_rgid = nullptr; s->ray_cap = 0;
      HIPOK(hipMalloc(&s->d_rays, total * 6 * sizeof(float)));
      HIPOK(hipMalloc(&s->d_rdist, total * sizeof(float)));
      HIPOK(hipMalloc(&s->d_rgid, total * sizeof(int)));
      s->ray_cap = total;
    }
    if (!s->d_gmask) HIPOK(hipMalloc(&s->d_gmask, m.ngeom * sizeof(int)));
    float *d_pnt = s->d_rays, *d_vec = d_pnt + total * 3;
    // the queued steps finish before the host buffers are reused
    HIPOK(hipStreamSynchronize(s->stream));
    // a few rays: both arrays in one copy, whose start costs more than moving them
    // together (200 envs x 30 rays, 144 KB: 75 us in two, 69 in one; 500 x 64,
    // 768 KB: 99 in two, 109 in one)
    size_t bytes = total * 3 * sizeof(float);
    if (2 * bytes <= RAYS_ONE_COPY) {
      s->h_rays.resize(total * 6);
      std::memcpy(s->h_rays.data(), pnt, bytes);
      std::memcpy(s->h_rays.data() + total * 3, vec, bytes);
      HIPOK(hipMemcpyAsync(d_pnt, s->h_rays.data(), 2 * bytes, hipMemcpyHostToDevice, s->stream));
    } else {
      HIPOK(hipMemcpyAsync(d_pnt, pnt, bytes, hipMemcpyHostToDevice, s->stream));
      HIPOK(hipMemcpyAsync(d_vec, vec, bytes, hipMemcpyHostToDevice, s->stream));
    }
    HIPOK(hipMemcpyAsync(s->d_gmask, mask.data(), mask.size() * sizeof(int), hipMemcpyHostToDevice, s->stream));
    if (s->use_gws)
      hipLaunchKernelGGL(k_raycast<1>, dim3(s->B), dim3(64), 0, s->stream, s->dm, s->L, s->d_qpos, s->d_rand,
                         s->nrand, d_pnt, d_vec, nray, s->d_gmask, s->d_rdist, s->d_rgid, s->B, s->d_gws);
    else
      hipLaunchKernelGGL(k_raycast<0>, dim3(s->B), dim3(64), s->lds_bytes, s->stream, s->dm, s->L, s->d_qpos,
                         s->d_rand, s->nrand, d_pnt, d_vec, nray, s->d_gmask, s->d_rdist, s->d_rgid, s->B, nullptr);
    HIPOK(hipGetLastError());
    HIPOK(hipMemcpyAsync(dist_out, s->d_rdist, total * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipMemcpyAsync(geomid_out, s->d_rgid, total * sizeof(int), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_raycast", e); return -1; }
}

MJMLX_API void mjmlx_batched_eval_state(const MjmlxBatchedSim* s) {
  if (s) hipStreamSynchronize(s->stream);
}

MJMLX_API void mjmlx_grad_step(const MjmlxModel*, const MjmlxData*, float*) {}
MJMLX_API void mjmlx_batched_grad_step(MjmlxBatchedSim*, float*) {}

MJMLX_API MjmlxCameraRenderer* mjmlx_camera_create(MjmlxBatchedSim*, int, int) {
  std::fprintf(stderr, "mjmlx_camera_create error: rendering is not part of the HIP engine\n");
  return nullptr;
}
MJMLX_API void mjmlx_camera_free(MjmlxCameraRenderer*) {}
MJMLX_API int mjmlx_camera_count(const MjmlxCameraRenderer*) { return 0; }
MJMLX_API int mjmlx_camera_render(MjmlxCameraRenderer*) { return -1; }
MJMLX_API int mjmlx_camera_draw_call_count(const MjmlxCameraRenderer*) { return 0; }
MJMLX_API int mjmlx_camera_get_rgb(MjmlxCameraRenderer*, uint8_t*) { return -1; }
MJMLX_API int mjmlx_camera_get_depth(MjmlxCameraRenderer*, float*) { return -1; }
MJMLX_API int mjmlx_camera_gpu_supported(const MjmlxCameraRenderer*) { return 0; }
MJMLX_API int mjmlx_camera_gpu_copy(MjmlxCameraRenderer*) { return -1; }
MJMLX_API int mjmlx_camera_gpu_export_fd(MjmlxCameraRenderer*, int, uint64_t*) { return -1; }

// ---- additions (mjmlx_hip.h)
MJMLX_API int mjmlx_batched_set_warmstart_mode(MjmlxBatchedSim* s, int mode) {
  if (!s || mode < 0 || mode > 3) return -1;
  if (mode >= 2 && !s->mlp) {
    std::fprintf(stderr, "mjmlx_batched_set_warmstart_mode error: modes 2 and 3 need mjmlx_batched_set_warmstart_mlp first\n");
    return -1;
  }
  try {
    s->ws_mode = mode;
    if (mode == 1) s->dm.disableflags |= mjk::DS_WARMSTART;
    else s->dm.disableflags &= ~mjk::DS_WARMSTART;
    upload_kparams(s);
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_set_warmstart_mode", e); return -1; }
}

MJMLX_API int mjmlx_batched_get_qacc_warmstart(const MjmlxBatchedSim* cs, float* out) {
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  if (!s || !out) return -1;
  try {
    HIPOK(hipMemcpyAsync(out, s->d_qws, (size_t)s->B * s->nv * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_get_qacc_warmstart", e); return -1; }
}

MJMLX_API int mjmlx_batched_set_qacc_warmstart(MjmlxBatchedSim* s, const float* in) {
  if (!s || !in) return -1;
  try {
    HIPOK(hipStreamSynchronize(s->stream));
    HIPOK(hipMemcpy(s->d_qws, in, (size_t)s->B * s->nv * sizeof(float), hipMemcpyHostToDevice));
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_set_qacc_warmstart", e); return -1; }
}

MJMLX_API int mjmlx_batched_solver_stats(const MjmlxBatchedSim* cs, int* niter, int* status, int* ncon, int* nefc) {
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  if (!s) return -1;
  try {
    size_t n = (size_t)s->B * sizeof(int);
    if (niter) HIPOK(hipMemcpyAsync(niter, s->d_niter, n, hipMemcpyDeviceToHost, s->stream));
    if (status) HIPOK(hipMemcpyAsync(status, s->d_status, n, hipMemcpyDeviceToHost, s->stream));
    if (ncon) HIPOK(hipMemcpyAsync(ncon, s->d_ncon, n, hipMemcpyDeviceToHost, s->stream));
    if (nefc) HIPOK(hipMemcpyAsync(nefc, s->d_nefc, n, hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_solver_stats", e); return -1; }
}

MJMLX_API int mjmlx_batched_set_launch(MjmlxBatchedSim* s, int persistent, int grid) {
  if (!s || grid < 0) return -1;
  if (persistent) {
    // the work-queue launch hung once on the GPU with no cause found yet; it
    // stays switched off until one is shown
    std::fprintf(stderr, "mjmlx_batched_set_launch error: the persistent work-queue launch is disabled\n");
    return -1;
  }
  s->persistent = 0;
  s->grid = grid;
  return 0;
}

MJMLX_API int mjmlx_batched_autotune(MjmlxBatchedSim* s, int steps, int* choice) {
  if (!s || steps < 1) return -1;
  try {
    if (s->lds_ok) {
      size_t B = s->B;
      // every device buffer the timed steps write: the state, the solver
      // statistics, the sensors (values and the accelerometers' history) and
      // the aux outputs; restored after the timing so that the sim continues
      // from the state it was tuned at
      std::vector<std::pair<void*, size_t>> live = {
          {s->d_qpos, B * std::max(1, s->nq) * sizeof(float)}, {s->d_qvel, B * std::max(1, s->nv) * sizeof(float)},
          {s->d_qws, B * std::max(1, s->nv) * sizeof(float)},  {s->d_ctrl, B * std::max(1, s->nu) * sizeof(float)},
          {s->d_niter, B * sizeof(int)}, {s->d_status, B * sizeof(int)}, {s->d_ncon, B * sizeof(int)},
          {s->d_nefc, B * sizeof(int)}};
      if (s->d_sensordata) {
        live.push_back({s->d_sensordata, B * s->model.nsensordata * sizeof(float)});
        live.push_back({s->d_sens_prev, B * ((size_t)s->dm.nsens_acc * 3 + 1) * sizeof(float)});
      }
      if (s->aux_on)
        for (int i = 0; i < 7; i++) live.push_back({s->d_aux[i], std::max<size_t>(1, s->aux_len(i)) * sizeof(float)});
      std::vector<void*> saved(live.size(), nullptr);
      for (size_t i = 0; i < live.size(); i++) {
        HIPOK(hipMalloc(&saved[i], live[i].second));
        HIPOK(hipMemcpyAsync(saved[i], live[i].first, live[i].second, hipMemcpyDeviceToDevice, s->stream));
      }
      auto restore = [&]() {
        for (size_t i = 0; i < live.size(); i++)
          HIPOK(hipMemcpyAsync(live[i].first, saved[i], live[i].second, hipMemcpyDeviceToDevice, s->stream));
      };
      bool had_gws = s->d_gws != nullptr;
      if (!s->d_gws) HIPOK(hipMalloc(&s->d_gws, B * s->L.total * sizeof(float)));
      hipEvent_t e0, e1;
      HIPOK(hipEventCreate(&e0));
      HIPOK(hipEventCreate(&e1));
      const bool can_compact = s->d_kpc != nullptr;
      // candidates: 0 LDS at 256 registers (two waves per SIMD), 1 device
      // memory, 2 LDS at 168 VGPRs (three waves per SIMD, some spills), 3 LDS
      // at 512 registers (one wave per SIMD), 4 device memory at 168 VGPRs,
      // and for models that fit them, 32 lanes per env: 5 at 256 registers, 6
      // at 168 VGPRs
      // and CHOICE_COMPACT: small LDS workspaces first, where the sim has them
      const int ncand = can_compact ? CHOICE_COMPACT + 1 : (s->half_ok ? 7 : 5);
      float ms[CHOICE_COMPACT + 1];
      std::fill(ms, ms + CHOICE_COMPACT + 1, 3.0e38f);
      auto pick = [&](int g) {
        s->compact = g == CHOICE_COMPACT;
        s->use_gws = g == 1 || g == 4 || g == CHOICE_COMPACT;
        s->high_occ = g == 2 || g == 4 || g == 6;
        s->big_regs = g == 3;
        s->half = g == 5 || g == 6;
      };
      mjk::StepIO io = make_io(s, nullptr, nullptr);
      // the device is drained first so that other work does not share the timing
      HIPOK(hipDeviceSynchronize());
      for (int rep = 0; rep < 3; rep++)
        for (int g = 0; g < ncand; g++) {
          if ((g == 5 || g == 6) && !s->half_ok) continue;
          pick(g);
          restore();
          HIPOK(hipEventRecord(e0, s->stream));
          for (int k = 0; k < steps; k++) launch_step(s, io, 4);
          HIPOK(hipEventRecord(e1, s->stream));
          HIPOK(hipGetLastError());
          HIPOK(hipEventSynchronize(e1));
          float t = 0.f;
          HIPOK(hipEventElapsedTime(&t, e0, e1));
          if (rep > 0) ms[g] = std::min(ms[g], t);  // the first round warms caches and code
        }
      int best = 0;
      for (int g = 1; g < ncand; g++)
        if (ms[g] < ms[best]) best = g;
      pick(best);
      restore();
      HIPOK(hipStreamSynchronize(s->stream));
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      for (void* p : saved) HIPOK(hipFree(p));
      if (!s->use_gws && !had_gws) { HIPOK(hipFree(s->d_gws)); s->d_gws = nullptr; }
    }
    if (choice) *choice = mjmlx_batched_variant(s);
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_autotune", e); return -1; }
}

MJMLX_API int mjmlx_batched_variant(const MjmlxBatchedSim* s) {
  if (!s) return -1;
  return s->compact ? CHOICE_COMPACT : step_variant(s);
}

MJMLX_API int mjmlx_batched_set_variant(MjmlxBatchedSim* s, int choice) {
  if (!s || choice < 0 || choice > CHOICE_COMPACT) return -1;
  if (choice == CHOICE_COMPACT && !s->d_kpc) return -1;
  // the full-size rerun takes device memory, as when the autotuner times it
  bool gws = choice == 1 || choice == 4 || choice == CHOICE_COMPACT, half = choice == 5 || choice == 6;
  if (!gws && !s->lds_ok) return -1;  // LDS variants: the workspace must fit a workgroup's LDS
  if (half && !s->half_ok) return -1;
  try {
    if (gws && !s->d_gws) HIPOK(hipMalloc(&s->d_gws, (size_t)s->B * s->L.total * sizeof(float)));
    s->use_gws = gws;
    s->high_occ = choice == 2 || choice == 4 || choice == 6;
    s->big_regs = choice == 3;
    s->half = half;
    s->compact = choice == CHOICE_COMPACT;
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_set_variant", e); return -1; }
}

MJMLX_API int mjmlx_batched_set_graph(MjmlxBatchedSim* s, int on) {
  if (!s) return -1;
  s->graph_on = on != 0;
  return 0;
}

MJMLX_API float mjmlx_batched_last_step_ms(const MjmlxBatchedSim* s) {
  if (!s || !s->timed) return 0.f;
  float ms = 0.f;
  if (hipEventSynchronize(s->ev1) != hipSuccess) return 0.f;
  if (hipEventElapsedTime(&ms, s->ev0, s->ev1) != hipSuccess) return 0.f;
  return ms;
}

MJMLX_API int mjmlx_batched_capacity(const MjmlxBatchedSim* s, int* maxcon, int* maxefc, int* lds_bytes) {
  if (!s) return -1;
  if (maxcon) *maxcon = s->L.maxcon;
  if (maxefc) *maxefc = s->L.maxefc;
  if (lds_bytes) *lds_bytes = (int)s->lds_bytes;
  return 0;
}

MJMLX_API int mjmlx_batched_debug_step(MjmlxBatchedSim* s, const float* ctrl, float* dump1, float* dump2) {
  if (!s) return -1;
  try {
    size_t need = (size_t)s->B * s->L.total;
    if (s->dump_cap < need) {
      if (s->d_dump1) hipFree(s->d_dump1);
      if (s->d_dump2) hipFree(s->d_dump2);
      s->d_dump1 = s->d_dump2 = nullptr;
      HIPOK(hipMalloc(&s->d_dump1, need * sizeof(float)));
      HIPOK(hipMalloc(&s->d_dump2, need * sizeof(float)));
      s->dump_cap = need;
    }
    upload_ctrl(s, ctrl);
    launch(s, 1, s->d_dump1, s->d_dump2);
    if (dump1) HIPOK(hipMemcpyAsync(dump1, s->d_dump1, need * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    if (dump2) HIPOK(hipMemcpyAsync(dump2, s->d_dump2, need * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_debug_step", e); return -1; }
}

// Per-stage cycle counts of one call (profiling builds only: compiled with
// MJK_PROFILE); out is unsigned long long[num_envs * 17]. Returns 0, or -1
// in builds without the instrumentation.
MJMLX_API int mjmlx_batched_profile_step(MjmlxBatchedSim* s, const float* ctrl, int nsub, unsigned long long* out) {
#if defined(MJK_PROFILE)
  if (!s || !out || nsub <= 0) return -1;
  try {
    unsigned long long* d = nullptr;
    size_t n = (size_t)s->B * mjk::KP_N;
    HIPOK(hipMalloc(&d, n * sizeof(unsigned long long)));
    upload_ctrl(s, ctrl);
    mjk::StepIO io = make_io(s, nullptr, nullptr);
    io.prof = d;
    launch_step(s, io, nsub);
    HIPOK(hipGetLastError());
    HIPOK(hipMemcpyAsync(out, d, n * sizeof(unsigned long long), hipMemcpyDeviceToHost, s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    (void)hipFree(d);
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_profile_step", e); return -1; }
#else
  (void)s; (void)ctrl; (void)nsub; (void)out;
  return -1;
#endif
}

MJMLX_API int mjmlx_batched_feature_dim(const MjmlxBatchedSim* s) { return s ? s->nfeat() : -1; }

MJMLX_API int mjmlx_batched_set_feature_mode(MjmlxBatchedSim* s, int mode) {
  if (!s || mode < 0 || mode > 1) return -1;
  if (mode != s->feat_mode) {
    s->feat_mode = mode;
    s->feat_valid = false;
    if (s->mlp) {
      s->mlp = nullptr;  // its input width no longer matches
      if (s->ws_mode >= 2) s->ws_mode = 0;
    }
  }
  return 0;
}

MJMLX_API int mjmlx_batched_set_warmstart_mlp(MjmlxBatchedSim* s, MjmlxMLP* mlp) {
  if (!s) return -1;
  if (!mlp) {
    s->mlp = nullptr;
    if (s->ws_mode >= 2) s->ws_mode = 0;
    return 0;
  }
  int nin = 0, nout = 0;
  mjmlx_mlp_dims(mlp, &nin, nullptr, &nout, nullptr);
  if (nin != s->nfeat() || nout != s->nv) {
    std::fprintf(stderr, "mjmlx_batched_set_warmstart_mlp error: network is %d -> %d, the model needs %d -> %d\n", nin,
                 nout, s->nfeat(), s->nv);
    return -1;
  }
  try {
    ensure_learned(s);
    // a network may have the address of a freed one, and a captured step its buffers
    s->g_mlp = nullptr;
    s->mlp = mlp;
    return 0;
  } catch (const std::exception& e) { report("mjmlx_batched_set_warmstart_mlp", e); return -1; }
}

MJMLX_API long mjmlx_batched_record(MjmlxBatchedSim* s, MjmlxMLP* mlp, const float* ctrl, int nsub) {
  if (!s || !mlp || nsub <= 0) return -1;
  int nin = 0, nout = 0;
  mjmlx_mlp_dims(mlp, &nin, nullptr, &nout, nullptr);
  if (nin != s->nfeat() || nout != s->nv) return -1;
  try {
    upload_ctrl(s, ctrl);
    return step_substeps(s, nsub, mlp);
  } catch (const std::exception& e) { report("mjmlx_batched_record", e); return -1; }
}

MJMLX_API int mjmlx_batched_get_features(const MjmlxBatchedSim* cs, float* out) {
  auto* s = const_cast<MjmlxBatchedSim*>(cs);
  if (!s || !out || !s->d_pred || !s->feat_valid) return -1;
  try {
    HIPOK(hipMemcpyAsync(out, s->d_feat[s->feat_cur], (size_t)s->B * s->nfeat() * sizeof(float), hipMemcpyDeviceToHost,
                         s->stream));
    HIPOK(hipStreamSynchronize(s->stream));
    return s->nfeat();
  } catch (const std::exception& e) { report("mjmlx_batched_get_features", e); return -1; }
}

MJMLX_API int mjmlx_batched_layout(const MjmlxBatchedSim* s, const char* name, int* off, int* len, int* kind) {
  if (!s || !name) return -1;
  if (std::strcmp(name, "total") == 0) { *off = 0; *len = s->L.total; *kind = 0; return 0; }
  for (auto& f : s->fields)
    if (std::strcmp(f.name, name) == 0) { *off = f.off; *len = f.len; *kind = f.kind; return 0; }
  return -1;
}

}  // extern "C"
