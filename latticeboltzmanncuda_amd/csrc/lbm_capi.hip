// C-ABI of liblbm_hip.so: context lifetime, host <-> device exchange,
// geometry upload, stage and step launches, readback.  Every call checks
// its arguments and HIP return codes and reports failures through an
// lbm_status plus a thread-local message (lbm_last_error).
//
// Host <-> device copies run on the context's stream and are followed by a
// synchronisation of that stream; step and stage launches are asynchronous.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <exception>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "lbm_internal.h"
#include "lbm_lattice.h"
#include "lbm_layout.h"
#include "lbm_store.h"
#include "lbm_box.h"
#include "lbm_march.h"
#include "lbm_sweep.h"

namespace lbm {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  g_last_error = std::string(what) + ": " + hipGetErrorString(e);
  return e == hipErrorOutOfMemory ? LBM_ERR_NOMEM : LBM_ERR_HIP;
}

int api_exception() noexcept {
  int code = LBM_ERR_INVALID;
  const char* msg = "internal error: unknown exception";
  try {
    throw;
  } catch (const std::bad_alloc&) {
    code = LBM_ERR_NOMEM;
    msg = "host allocation failed";
  } catch (const std::exception& e) {
    msg = e.what();
  } catch (...) {
  }
  try {
    g_last_error = msg;
  } catch (...) {
    // no memory for the message either: keep the previous one
  }
  return code;
}

namespace {

// Fills the per-direction constants of lattice L in precision C.  The
// products are formed in C from the configured float values, as the
// kernels formed them before they were hoisted.
template <class L, class C>
void fill_coef(const StdParams& p, StepCoef<C>& k) {
  const C omega = (C)1 / (C)p.tau;
  const C guo = (C)1 - (C)0.5 * omega;
  k.omega = omega;
  for (int a = 0; a < 3; ++a) {
    k.force[a] = (C)p.force[a];
    k.half_force[a] = (C)0.5 * (C)p.force[a];
  }
  k.forced = p.force[0] != 0.0f || p.force[1] != 0.0f || p.force[2] != 0.0f;
  for (int i = 0; i < L::Q; ++i) {
    const int* e = L::E[i];
    const C w = (C)L::W[i];
    const C eF = (C)e[0] * k.force[0] + (C)e[1] * k.force[1] + (C)e[2] * k.force[2];
    k.gw[i] = guo * w;
    k.gf3[i] = k.gw[i] * ((C)3 * eF);
    k.gf9[i] = k.gw[i] * ((C)9 * eF);
    k.lid[i] = (C)0;
    if (p.lid_axis >= 0 && e[p.lid_axis] == -p.lid_sign) {
      // a link of direction i whose source node lies beyond the moving face
      const C eu = (C)e[0] * (C)p.lid_u[0] + (C)e[1] * (C)p.lid_u[1] + (C)e[2] * (C)p.lid_u[2];
      k.lid[i] = (C)6 * w * (C)p.wall_rho * eu;
    }
  }
}

// cf in FP16 stored units: exact, as the scale is a power of two
template <class L>
void fill_coef_units(const StepCoef<float>& k, float scale, StepCoef<float>& u) {
  u = k;
  for (int a = 0; a < 3; ++a) u.half_force[a] = k.half_force[a] * scale;
  for (int i = 0; i < L::Q; ++i) {
    u.lid[i] = k.lid[i] * scale;
    u.gw[i] = k.gw[i] * scale;
    u.gf3[i] = k.gf3[i] * scale;
    u.gf9[i] = k.gf9[i] * scale;
  }
}

template <class L>
void fill_coefs(StdParams& p) {
  fill_coef<L, float>(p, p.cf);
  fill_coef<L, double>(p, p.cd);
  fill_coef_units<L>(p.cf, 1.0f / Store<LBM_STORE_F16>::kUnit, p.ch);
}

}  // namespace

StdParams make_std_params(const lbm_config& cfg) {
  StdParams p{};
  p.tau = cfg.tau;
  for (int a = 0; a < 3; ++a) {
    p.force[a] = cfg.force[a];
    p.lid_u[a] = cfg.lid_u[a];
  }
  p.lid_axis = cfg.lid_face >= 0 ? cfg.lid_face / 2 : -1;
  p.lid_sign = cfg.lid_face >= 0 ? (cfg.lid_face % 2 ? 1 : -1) : 0;
  p.wall_rho = cfg.wall_rho;
  switch (cfg.lattice) {
    case 9:
      fill_coefs<Lat<9>>(p);
      break;
    case 19:
      fill_coefs<Lat<19>>(p);
      break;
    default:
      fill_coefs<Lat<27>>(p);
      break;
  }
  return p;
}

double cell_reynolds(const lbm_config& cfg) {
  const double nu = ((double)cfg.tau - 0.5) / 3.0;
  const double uw = std::sqrt((double)cfg.lid_u[0] * cfg.lid_u[0] +
                              (double)cfg.lid_u[1] * cfg.lid_u[1] +
                              (double)cfg.lid_u[2] * cfg.lid_u[2]);
  const double F = std::sqrt((double)cfg.force[0] * cfg.force[0] +
                             (double)cfg.force[1] * cfg.force[1] +
                             (double)cfg.force[2] * cfg.force[2]);
  // narrowest walled extent (axes of one node carry no flow)
  const int32_t ext[3] = {cfg.nx, cfg.ny, cfg.nz};
  int32_t walled = 0, widest = 1;
  for (int a = 0; a < 3; ++a) {
    if (ext[a] < 2) continue;
    widest = std::max(widest, ext[a]);
    if (!cfg.periodic[a]) walled = walled ? std::min(walled, ext[a]) : ext[a];
  }
  const double W = walled ? walled : widest;
  const double U = std::max(cfg.lid_face >= 0 ? uw : 0.0, F * W * W / (8.0 * nu));
  return U / nu;
}

int64_t estimate_ctx_bytes(const lbm_config& cfg) {
  const uint64_t n = (uint64_t)cfg.nx * cfg.ny * cfg.nz;
  int64_t b = 2 * (int64_t)(population_elems(cfg.lattice, n) * storage_bytes(cfg.storage));
  if (cfg.mode == LBM_MODE_STANDARD)
    b += (has_mask16(cfg) ? 6 : 4) * (int64_t)n + 4 * (int64_t)((n + 15) / 16);
  else
    b += (int64_t)n;
  b += 4 * 1024 * 8 * 4 + 64;  // reduction scratch, force register
  return b;
}

namespace {

// Scoped device allocation for staging buffers.
struct DevBuf {
  void* p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  int alloc(size_t bytes) {
    hipError_t e = hipMalloc(&p, bytes ? bytes : 1);
    if (e != hipSuccess) {
      p = nullptr;
      return hip_fail(e, "hipMalloc(staging)");
    }
    return LBM_OK;
  }
};

int check_ctx(const lbm_ctx* c) {
  if (!c) return fail(LBM_ERR_INVALID, "null context");
  return LBM_OK;
}

int need_mode(const lbm_ctx* c, int mode, const char* what) {
  if (c->cfg.mode != mode)
    return fail(LBM_ERR_STATE,
                std::string(what) + " needs " +
                    (mode == LBM_MODE_REFERENCE ? "reference" : "standard") +
                    " mode");
  return LBM_OK;
}

int dev_alloc(lbm_ctx* c, void** p, size_t bytes, const char* what) {
  hipError_t e = hipMalloc(p, bytes ? bytes : 1);
  if (e != hipSuccess) {
    *p = nullptr;
    return hip_fail(e, what);
  }
  c->device_bytes += (int64_t)bytes;
  return LBM_OK;
}

void dev_free(lbm_ctx* c, void** p, size_t bytes) {
  if (*p) {
    (void)hipFree(*p);
    c->device_bytes -= (int64_t)bytes;
  }
  *p = nullptr;
}

int sync(lbm_ctx* c) {
  LBM_HIP(hipStreamSynchronize(c->stream));
  return LBM_OK;
}

// Solid nodes are never written by a standard step, so after a host
// upload both population buffers are made equal.
int mirror_buffers(lbm_ctx* c) {
  const size_t fbytes = population_elems(c->q, c->grid.n) * c->elem;
  LBM_HIP(hipMemcpyAsync(c->f[c->cur ^ 1], c->f[c->cur], fbytes,
                         hipMemcpyDeviceToDevice, c->stream));
  return LBM_OK;
}

int h2d(lbm_ctx* c, void* dst, const void* src, size_t bytes) {
  return copy_to_device(dst, src, bytes, c->stream);
}

int d2h(lbm_ctx* c, void* dst, const void* src, size_t bytes) {
  const HostPiece p{dst, bytes};
  return copy_to_host(src, &p, 1, c->stream);
}

int validate_config(const lbm_config* cfg) {
  if (!cfg) return fail(LBM_ERR_INVALID, "null config");
  if (cfg->nx < 1 || cfg->ny < 1 || cfg->nz < 1)
    return fail(LBM_ERR_INVALID, "lattice extents must be >= 1");
  // the kernels multiply coordinates and extents with 24-bit multiplies
  if (cfg->nx >= (1 << 24) || cfg->ny >= (1 << 24) || cfg->nz >= (1 << 24))
    return fail(LBM_ERR_UNSUPPORTED, "lattice extents must be below 2^24");
  const uint64_t n = (uint64_t)cfg->nx * cfg->ny * cfg->nz;
  if (cfg->lattice != 9 && cfg->lattice != 19 && cfg->lattice != 27)
    return fail(LBM_ERR_INVALID, "lattice must be 9, 19 or 27");
  if (population_elems(cfg->lattice, n) >= (1ull << 31))
    return fail(LBM_ERR_UNSUPPORTED,
                "lattice too large for 32-bit population indices");
  if (cfg->lattice == 9 && cfg->nz != 1)
    return fail(LBM_ERR_INVALID, "D2Q9 needs nz == 1");
  if (storage_bytes(cfg->storage) == 0)
    return fail(LBM_ERR_INVALID, "unknown storage type");
  if (cfg->mode != LBM_MODE_STANDARD && cfg->mode != LBM_MODE_REFERENCE)
    return fail(LBM_ERR_INVALID, "unknown mode");
  if (cfg->mode == LBM_MODE_REFERENCE &&
      (cfg->lattice != 27 || cfg->storage != LBM_STORE_F32))
    return fail(LBM_ERR_UNSUPPORTED, "reference mode is D3Q27 with F32 storage");
  if (!(cfg->tau > 0.0f))
    return fail(LBM_ERR_INVALID, "tau must be positive");
  if (cfg->mode == LBM_MODE_STANDARD && !(cfg->tau > 0.5f))
    return fail(LBM_ERR_INVALID, "standard BGK needs tau > 1/2");
  for (int a = 0; a < 3; ++a)
    if (!std::isfinite(cfg->force[a]) || !std::isfinite(cfg->lid_u[a]))
      return fail(LBM_ERR_INVALID, "body force and wall velocity must be finite");
  if (!std::isfinite(cfg->wall_rho)) return fail(LBM_ERR_INVALID, "wall density must be finite");
  if (cfg->lattice == 9 && cfg->force[2] != 0.0f)
    return fail(LBM_ERR_INVALID, "D2Q9 has no z axis: the body force's z component must be 0");
  if (cfg->lid_face < -1 || cfg->lid_face > 5)
    return fail(LBM_ERR_INVALID, "lid_face must be -1..5");
  if (cfg->lid_face >= 0) {
    const int ax = cfg->lid_face / 2;
    if (cfg->periodic[ax])
      return fail(LBM_ERR_INVALID, "moving wall on a periodic axis");
    if (cfg->lattice == 9 && ax == 2)
      return fail(LBM_ERR_INVALID, "D2Q9 has no z faces");
  }
  return LBM_OK;
}

Grid make_grid(const lbm_config& cfg) {
  Grid g{};
  g.nx = (uint32_t)cfg.nx;
  g.ny = (uint32_t)cfg.ny;
  g.nz = (uint32_t)cfg.nz;
  g.n = g.nx * g.ny * g.nz;
  g.dz = make_magic(g.nz);
  g.dy = make_magic(g.ny);
  g.flags = wrap_bits(cfg.periodic);
  return g;
}

// The geometry tables, rebuilt after a change of flags or records.
int rebuild_special(lbm_ctx* c) {
  if (!c->special_dirty) return LBM_OK;
  if (int rc = build_receivers(c)) return rc;
  c->special_dirty = false;
  return LBM_OK;
}

// From this many steps on one launch more is worth the smaller ones (about
// 1 us of host time each against 3 to 4 us).
constexpr int kPutSteps = 16;

// How a call of n steps of a lattice is launched: `kernel` (lbm_step_kernel)
// takes the launches of several steps or, where there are none, the single
// ones; launches[k]: how many take k steps each, the long ones first.
struct StepPlan {
  int kernel = LBM_STEP_NODE;
  int launches[LBM_MAX_LAUNCH_STEPS + 1] = {};
  MarchPlan march{};
  SweepPlan sweep{};
};

// As many launches, odd or even, as there are steps: a caller who captures
// them finds the state in the same buffer as after single steps.
StepPlan plan_steps(int q, int storage, const Grid& g, int n) {
  StepPlan p;
  if (n <= 1) {
    p.kernel = std_single_kernel(q, storage, g);
    p.launches[1] = n;
    return p;
  }
  const int box = std_box_steps(q, storage, g);
  if (box || std_sweeps(q, storage, g)) {
    p.kernel = box ? LBM_STEP_BOX : LBM_STEP_SWEEP;
    // boxes of 8 steps come in pairs
    if (box == 8) p.launches[8] = n / 16 * 2;
    split_steps(n - 8 * p.launches[8], box ? box_costs(storage, g) : sweep_costs(storage),
                p.launches);
    if (!box)
      p.sweep = sweep_plan(g, sweep_chunk_rows(1, [&](size_t) -> const Grid& { return g; }, storage));
  } else if (n >= 4 && std_marches(q, storage, g, &p.march)) {
    p.kernel = LBM_STEP_MARCH;
    p.launches[2] = n / 4 * 2;
    p.launches[1] = n % 4;
  } else {
    p.launches[1] = n;
  }
  if (p.launches[1] == n) p.kernel = std_single_kernel(q, storage, g);
  return p;
}

int step_standard(lbm_ctx* c, int n) {
  const StdParams p = make_std_params(c->cfg);
  const int storage = device_storage(c->cfg.mode, c->cfg.storage);
  const StepPlan plan = plan_steps(c->q, storage, c->grid, n);
  // the constants as they are now, for this call's launches alone: whoever
  // changes them, or captures the call, finds what a launch with them as
  // arguments would do
  const void* coef = nullptr;
  if (n >= kPutSteps && std_takes_coef(c->q, storage, c->grid)) {
    if (int rc = launch_put_coef(c->q, storage, p, c->coef, c->stream)) return rc;
    coef = c->coef;
  }
  for (int k = LBM_MAX_LAUNCH_STEPS; k > 0; --k)
    for (int s = 0; s < plan.launches[k]; ++s) {
      const void* A = c->f[c->cur];
      void* B = c->f[c->cur ^ 1];
      int rc;
      if (k == 1)
        rc = launch_std_step(c->q, storage, c->grid, A, B, c->mask, c->cls, p,
                             (int)(c->steps_done & 1), c->stream, coef);
      else if (plan.kernel == LBM_STEP_MARCH)
        rc = launch_std_march(storage, c->grid, plan.march, A, B, c->mask, p, c->stream);
      else if (plan.kernel == LBM_STEP_BOX)
        rc = launch_std_box(k, storage, c->grid, A, B, c->mask, c->cls, p, c->stream);
      else
        rc = launch_std_sweep(k, storage, c->grid, plan.sweep, A, B, c->mask, p, c->stream);
      if (rc) return rc;
      c->cur ^= 1;
      c->steps_done += k;
    }
  return LBM_OK;
}

int step_reference_fused(lbm_ctx* c, int n) {
  for (int s = 0; s < n; ++s) {
    int rc = launch_ref_stream_collide(c->grid, (const float*)c->f[c->cur],
                                       (float*)c->f[c->cur ^ 1], c->cfg.tau,
                                       c->stream);
    if (rc) return rc;
    c->cur ^= 1;
  }
  return LBM_OK;
}

int reflect(lbm_ctx* c, int with_force) {
  int rc = rebuild_special(c);
  if (rc) return rc;
  return launch_ref_reflect(c->grid, (float*)c->f[c->cur], c->nspecial,
                            c->special, c->special_rec, c->flags, c->rec_dirs,
                            c->rec_w, c->force_partials,
                            ref_reflect_blocks(c->nspecial),
                            with_force ? c->force : nullptr, c->stream);
}

// The reference's main loop S -> R -> C -> F (LatticeBoltzmannCuda.cpp:
// 85-93), one fused pass per step.
int step_reference_full(lbm_ctx* c, int n, int with_force) {
  int rc = rebuild_special(c);
  if (rc) return rc;
  const bool geom = c->ref_geom;
  for (int s = 0; s < n; ++s) {
    if ((rc = launch_ref_step_full(c->grid, (const float*)c->f[c->cur], (float*)c->f[c->cur ^ 1],
                                   c->cfg.tau, c->flow, geom ? c->ref_cls : nullptr,
                                   c->ref_inmask, c->ref_rxbase, c->ref_ngrp, c->ref_gsrc,
                                   c->ref_gbeg, c->ref_gid, c->ref_gsum, c->ref_nent, c->ref_eidx, c->ref_keep, c->ref_ew,
                                   c->ref_es, geom && with_force ? c->ref_partials : nullptr,
                                   geom && with_force ? c->force : nullptr, c->cur, c->stream)))
      return rc;
    c->cur ^= 1;
  }
  return LBM_OK;
}

// The same loop as separate stage passes (stream A -> B, reflect in place,
// collide + flow in place): the stage kernels the fused pass must match.
int step_reference_staged(lbm_ctx* c, int n, int with_force) {
  int rc = rebuild_special(c);
  if (rc) return rc;
  for (int s = 0; s < n; ++s) {
    if ((rc = launch_ref_stream(c->grid, (const float*)c->f[c->cur],
                                (float*)c->f[c->cur ^ 1], c->stream)))
      return rc;
    c->cur ^= 1;
    if ((rc = reflect(c, with_force))) return rc;
    if ((rc = launch_ref_collide(c->grid, (float*)c->f[c->cur], c->cfg.tau,
                                 &c->flow, c->stream)))
      return rc;
  }
  return LBM_OK;
}

}  // namespace

int check_config(const lbm_config* cfg) { return validate_config(cfg); }

int read_moments(lbm_ctx* c, void* stage, float* rho, float* u, bool plain) {
  const size_t N = c->grid.n;
  float* dr = rho ? (float*)stage : nullptr;
  float* du = u ? (float*)stage + (rho ? N : 0) : nullptr;
  int rc;
  if (c->cfg.mode == LBM_MODE_REFERENCE)
    rc = launch_ref_moments(c->grid, (const float*)c->f[c->cur], dr, du, c->stream);
  else
    rc = launch_std_moments(c->q, device_storage(c->cfg.mode, c->cfg.storage), c->grid,
                            c->f[c->cur], c->mask, c->cfg.force, dr, du, c->stream);
  if (rc) return rc;
  // rho and u lie side by side
  const HostPiece out[2] = {{rho, rho ? sizeof(float) * N : 0}, {u, u ? sizeof(float) * 3 * N : 0}};
  return plain ? copy_to_host_plain(stage, out, 2, c->stream)
               : copy_to_host(stage, out, 2, c->stream);
}

}  // namespace lbm

using namespace lbm;

extern "C" const char* lbm_last_error(void) { return g_last_error.c_str(); }

extern "C" int lbm_abi_version(void) { return LBM_ABI_VERSION; }

// The entry points of include/lbm.h; lbm_exports.hip exports each one
// with C linkage behind the exception boundary.
namespace lbm {
namespace api {

int lbm_device_info(int* device_count, char* name, size_t name_len) {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) return hip_fail(e, "hipGetDeviceCount");
  if (device_count) *device_count = n;
  if (name && name_len) {
    name[0] = 0;
    if (n > 0) {
      hipDeviceProp_t prop;
      LBM_HIP(hipGetDeviceProperties(&prop, 0));
      std::snprintf(name, name_len, "%s (%s, %d CUs)", prop.name,
                    prop.gcnArchName, prop.multiProcessorCount);
    }
  }
  return LBM_OK;
}

int lbm_create(const lbm_config* cfg, void* stream, lbm_ctx** out) {
  if (!out) return fail(LBM_ERR_INVALID, "null output handle");
  *out = nullptr;
  int rc = validate_config(cfg);
  if (rc) return rc;
  lbm_ctx* c = new (std::nothrow) lbm_ctx();
  if (!c) return fail(LBM_ERR_NOMEM, "host allocation of context");
  c->cfg = *cfg;
  c->q = cfg->lattice;
  c->elem = storage_bytes(cfg->storage);
  c->grid = make_grid(*cfg);
  const Grid& g = c->grid;
  c->flow.kind = LBM_FLOW_NONE;
  auto bail = [&](int code) {
    lbm_destroy(c);
    return code;
  };
  hipError_t e = hipGetDevice(&c->device);
  if (e != hipSuccess) return bail(hip_fail(e, "hipGetDevice"));
  if (stream) {
    c->stream = (hipStream_t)stream;
  } else {
    e = hipStreamCreate(&c->stream);
    if (e != hipSuccess) return bail(hip_fail(e, "hipStreamCreate"));
    c->own_stream = true;
  }
  if ((e = hipEventCreate(&c->ev0)) != hipSuccess ||
      (e = hipEventCreate(&c->ev1)) != hipSuccess)
    return bail(hip_fail(e, "hipEventCreate"));
  const size_t fbytes = population_elems(c->q, g.n) * c->elem;
  for (int k = 0; k < 2; ++k) {
    if ((rc = dev_alloc(c, &c->f[k], fbytes, "hipMalloc(populations)")))
      return bail(rc);
    if ((e = hipMemsetAsync(c->f[k], 0, fbytes, c->stream)) != hipSuccess)
      return bail(hip_fail(e, "hipMemsetAsync(populations)"));
  }
  if ((rc = dev_alloc(c, (void**)&c->force, 3 * sizeof(float), "hipMalloc(force)")))
    return bail(rc);
  if ((e = hipMemsetAsync(c->force, 0, 3 * sizeof(float), c->stream)) != hipSuccess)
    return bail(hip_fail(e, "hipMemsetAsync(force)"));
  c->red_cap = (int)std::min<uint32_t>(1024u, (g.n + 255) / 256);
  if ((rc = dev_alloc(c, (void**)&c->red, sizeof(double) * 4 * c->red_cap, "hipMalloc(reduction)")))
    return bail(rc);
  // the sums, and room for the step constants behind them
  if ((rc = dev_alloc(c, (void**)&c->red_out, 4 * sizeof(double) + kCoefBytes, "hipMalloc(reduction)")))
    return bail(rc);
  c->coef = (char*)c->red_out + 4 * sizeof(double);
  if (cfg->mode == LBM_MODE_STANDARD) {
    if ((rc = dev_alloc(c, (void**)&c->mask, (has_mask16(*cfg) ? 6 : 4) * (size_t)g.n,
                        "hipMalloc(mask)")))
      return bail(rc);
    if ((rc = dev_alloc(c, (void**)&c->cls, sizeof(uint32_t) * ((g.n + 15) / 16), "hipMalloc(class map)")))
      return bail(rc);
    if ((rc = launch_build_mask(c->q, g, nullptr, cfg->periodic, cfg->lid_face,
                                c->mask, c->cls, c->stream)) ||
        (has_mask16(*cfg) && (rc = launch_mask16(g, c->mask, c->stream))))
      return bail(rc);
  } else {
    if ((rc = dev_alloc(c, (void**)&c->flags, g.n, "hipMalloc(flags)")))
      return bail(rc);
    if ((e = hipMemsetAsync(c->flags, 0, g.n, c->stream)) != hipSuccess)
      return bail(hip_fail(e, "hipMemsetAsync(flags)"));
  }
  if ((rc = sync(c))) return bail(rc);
  transfer_context(1);
  c->counted = true;
  *out = c;
  return LBM_OK;
}

int lbm_destroy(lbm_ctx* c) {
  if (!c) return LBM_OK;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (void* p : {c->f[0], c->f[1], (void*)c->mask, (void*)c->cls, (void*)c->flags,
                  (void*)c->rec_node, (void*)c->rec_dirs, (void*)c->rec_w,
                  (void*)c->flow_mask, (void*)c->force, (void*)c->red, (void*)c->red_out,
                  c->ref_tables, c->stage})
    if (p) (void)hipFree(p);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  if (c->own_stream && c->stream) (void)hipStreamDestroy(c->stream);
  if (c->counted) transfer_context(-1);
  delete c;
  return LBM_OK;
}

int lbm_get_config(const lbm_ctx* c, lbm_config* out) {
  if (int rc = check_ctx(c)) return rc;
  if (!out) return fail(LBM_ERR_INVALID, "null output");
  *out = c->cfg;
  return LBM_OK;
}

int64_t lbm_node_count(const lbm_ctx* c) { return c ? (int64_t)c->grid.n : -1; }

int64_t lbm_device_bytes(const lbm_ctx* c) { return c ? c->device_bytes : -1; }

double lbm_cell_reynolds(const lbm_config* cfg) {
  if (int rc = validate_config(cfg)) return -(double)rc;
  if (cfg->mode != LBM_MODE_STANDARD)
    return -(double)fail(LBM_ERR_STATE, "lbm_cell_reynolds needs a standard-mode configuration");
  return cell_reynolds(*cfg);
}

int lbm_set_tau(lbm_ctx* c, float tau) {
  if (int rc = check_ctx(c)) return rc;
  if (!(tau > 0.0f) || (c->cfg.mode == LBM_MODE_STANDARD && !(tau > 0.5f)))
    return fail(LBM_ERR_INVALID, "tau out of range");
  c->cfg.tau = tau;
  ++c->params_version;
  return LBM_OK;
}

int lbm_set_body_force(lbm_ctx* c, const float force[3]) {
  if (int rc = check_ctx(c)) return rc;
  if (!force) return fail(LBM_ERR_INVALID, "null force");
  for (int a = 0; a < 3; ++a)
    if (!std::isfinite(force[a])) return fail(LBM_ERR_INVALID, "body force must be finite");
  if (c->cfg.lattice == 9 && force[2] != 0.0f)
    return fail(LBM_ERR_INVALID, "D2Q9 has no z axis: the body force's z component must be 0");
  for (int a = 0; a < 3; ++a) c->cfg.force[a] = force[a];
  ++c->params_version;
  return LBM_OK;
}

int lbm_synchronize(lbm_ctx* c) {
  if (int rc = check_ctx(c)) return rc;
  return sync(c);
}

int lbm_upload_points(lbm_ctx* c, const lbm_lattice_point* pts, int64_t count) {
  if (int rc = check_ctx(c)) return rc;
  if (!pts) return fail(LBM_ERR_INVALID, "null points");
  if (count != (int64_t)c->grid.n)
    return fail(LBM_ERR_INVALID, "point count does not match the lattice");
  DevBuf st;
  const size_t bytes = sizeof(lbm_lattice_point) * (size_t)count;
  int rc;
  if ((rc = st.alloc(bytes))) return rc;
  if ((rc = h2d(c, st.p, pts, bytes))) return rc;
  const bool ref = c->cfg.mode == LBM_MODE_REFERENCE;
  // whether any node's flags change is found on the GPU while they are
  // written: the geometry tables stay where none does
  DevBuf changed;
  int any = 0;
  if (ref) {
    if ((rc = changed.alloc(sizeof any))) return rc;
    LBM_HIP(hipMemsetAsync(changed.p, 0, sizeof any, c->stream));
  }
  if ((rc = launch_points_in(c->q, device_storage(c->cfg.mode, c->cfg.storage), c->grid,
                             (const lbm_lattice_point*)st.p, c->f[c->cur],
                             ref ? c->flags : nullptr, (int*)changed.p, c->stream)))
    return rc;
  if ((rc = mirror_buffers(c))) return rc;
  if (!ref) return sync(c);
  if ((rc = d2h(c, &any, changed.p, sizeof any))) return rc;
  if (any) c->special_dirty = true;
  return LBM_OK;
}

int lbm_download_points(lbm_ctx* c, lbm_lattice_point* pts, int64_t count) {
  if (int rc = check_ctx(c)) return rc;
  if (!pts) return fail(LBM_ERR_INVALID, "null points");
  if (count != (int64_t)c->grid.n)
    return fail(LBM_ERR_INVALID, "point count does not match the lattice");
  DevBuf st;
  const size_t bytes = sizeof(lbm_lattice_point) * (size_t)count;
  int rc;
  if ((rc = st.alloc(bytes))) return rc;
  if ((rc = launch_points_out(c->q, device_storage(c->cfg.mode, c->cfg.storage), c->grid, c->f[c->cur],
                              c->flags, (lbm_lattice_point*)st.p, c->stream)))
    return rc;
  return d2h(c, pts, st.p, bytes);
}

static int set_pops(lbm_ctx* c, const void* f, int is_f64) {
  if (int rc = check_ctx(c)) return rc;
  if (!f) return fail(LBM_ERR_INVALID, "null populations");
  const size_t bytes = (size_t)c->q * c->grid.n * (is_f64 ? 8 : 4);
  DevBuf st;
  int rc;
  if ((rc = st.alloc(bytes))) return rc;
  if ((rc = h2d(c, st.p, f, bytes))) return rc;
  if ((rc = launch_convert_in(c->q, device_storage(c->cfg.mode, c->cfg.storage), c->grid, st.p, is_f64,
                              c->f[c->cur], c->stream)))
    return rc;
  if ((rc = mirror_buffers(c))) return rc;
  return sync(c);
}

static int get_pops(lbm_ctx* c, void* f, int is_f64) {
  if (int rc = check_ctx(c)) return rc;
  if (!f) return fail(LBM_ERR_INVALID, "null populations");
  const size_t bytes = (size_t)c->q * c->grid.n * (is_f64 ? 8 : 4);
  DevBuf st;
  int rc;
  if ((rc = st.alloc(bytes))) return rc;
  if ((rc = launch_convert_out(c->q, device_storage(c->cfg.mode, c->cfg.storage), c->grid, c->f[c->cur],
                               st.p, is_f64, c->stream)))
    return rc;
  return d2h(c, f, st.p, bytes);
}

int lbm_set_populations_f32(lbm_ctx* c, const float* f) { return set_pops(c, f, 0); }
int lbm_get_populations_f32(lbm_ctx* c, float* f) { return get_pops(c, f, 0); }
int lbm_set_populations_f64(lbm_ctx* c, const double* f) { return set_pops(c, f, 1); }
int lbm_get_populations_f64(lbm_ctx* c, double* f) { return get_pops(c, f, 1); }

int lbm_init_equilibrium(lbm_ctx* c, const double* rho, const double* u) {
  if (int rc = check_ctx(c)) return rc;
  const size_t N = c->grid.n;
  DevBuf dr, du;
  int rc;
  if (rho) {
    if ((rc = dr.alloc(sizeof(double) * N))) return rc;
    if ((rc = h2d(c, dr.p, rho, sizeof(double) * N))) return rc;
  }
  if (u) {
    if ((rc = du.alloc(sizeof(double) * 3 * N))) return rc;
    if ((rc = h2d(c, du.p, u, sizeof(double) * 3 * N))) return rc;
  }
  if ((rc = launch_init_eq(c->q, device_storage(c->cfg.mode, c->cfg.storage), c->grid, (const double*)dr.p,
                           (const double*)du.p, c->f[c->cur], c->stream)))
    return rc;
  if ((rc = mirror_buffers(c))) return rc;
  return sync(c);
}

int lbm_upload_solid(lbm_ctx* c, const uint8_t* solid) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_STANDARD, "lbm_upload_solid")) return rc;
  DevBuf ds;
  int rc;
  bool any_solid = false;
  if (solid) {
    if ((rc = ds.alloc(c->grid.n))) return rc;
    if ((rc = h2d(c, ds.p, solid, c->grid.n))) return rc;
    for (uint32_t n = 0; n < c->grid.n && !any_solid; ++n) any_solid = solid[n] != 0;
  }
  c->grid.flags = (c->grid.flags & ~kReadMasks) | (any_solid ? kReadMasks : 0u);
  ++c->params_version;
  if ((rc = launch_build_mask(c->q, c->grid, (const uint8_t*)ds.p,
                              c->cfg.periodic, c->cfg.lid_face, c->mask,
                              c->cls, c->stream)) ||
      (has_mask16(c->cfg) && (rc = launch_mask16(c->grid, c->mask, c->stream))))
    return rc;
  return sync(c);
}

int lbm_get_mask(lbm_ctx* c, uint32_t* mask) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_STANDARD, "lbm_get_mask")) return rc;
  if (!mask) return fail(LBM_ERR_INVALID, "null mask");
  return d2h(c, mask, c->mask, sizeof(uint32_t) * c->grid.n);
}

int lbm_upload_flags(lbm_ctx* c, const uint8_t* flags) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_upload_flags")) return rc;
  if (!flags) return fail(LBM_ERR_INVALID, "null flags");
  c->special_dirty = true;
  return h2d(c, c->flags, flags, c->grid.n);
}

int lbm_get_flags(lbm_ctx* c, uint8_t* flags) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_get_flags")) return rc;
  if (!flags) return fail(LBM_ERR_INVALID, "null flags");
  return d2h(c, flags, c->flags, c->grid.n);
}

int lbm_upload_reflections(lbm_ctx* c, int32_t count, const int32_t* node,
                           const uint32_t* dirs, const float* weights) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_upload_reflections"))
    return rc;
  if (count < 0 || (count > 0 && (!node || !dirs || !weights)))
    return fail(LBM_ERR_INVALID, "bad reflection records");
  for (int32_t r = 0; r < count; ++r)
    if (node[r] < 0 || (uint32_t)node[r] >= c->grid.n)
      return fail(LBM_ERR_INVALID, "reflection record node out of range");
  const size_t old = (size_t)std::max(c->nrec, 1);
  dev_free(c, (void**)&c->rec_node, sizeof(int32_t) * old);
  dev_free(c, (void**)&c->rec_dirs, sizeof(uint32_t) * 14 * old);
  dev_free(c, (void**)&c->rec_w, sizeof(float) * 81 * old);
  c->nrec = 0;
  c->special_dirty = true;
  const size_t m = (size_t)std::max(count, 1);
  int rc;
  if ((rc = dev_alloc(c, (void**)&c->rec_node, sizeof(int32_t) * m, "hipMalloc(records)")) ||
      (rc = dev_alloc(c, (void**)&c->rec_dirs, sizeof(uint32_t) * 14 * m, "hipMalloc(records)")) ||
      (rc = dev_alloc(c, (void**)&c->rec_w, sizeof(float) * 81 * m, "hipMalloc(records)")))
    return rc;
  if (count > 0) {
    if ((rc = h2d(c, c->rec_node, node, sizeof(int32_t) * count)) ||
        (rc = h2d(c, c->rec_dirs, dirs, sizeof(uint32_t) * 14 * count)) ||
        (rc = h2d(c, c->rec_w, weights, sizeof(float) * 81 * count)))
      return rc;
  }
  c->nrec = count;
  // the reflection records usually complete the geometry: build the fused
  // step's receiver tables now rather than in the first step (a later flag
  // change marks them for rebuilding again)
  return rebuild_special(c);
}

int lbm_set_flow(lbm_ctx* c, int kind, const int32_t* params,
                 const float* induced, const uint8_t* mask) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_set_flow")) return rc;
  if (kind < LBM_FLOW_NONE || kind > LBM_FLOW_MASK)
    return fail(LBM_ERR_INVALID, "unknown flow kind");
  if (kind != LBM_FLOW_NONE && !induced)
    return fail(LBM_ERR_INVALID, "null induced flow");
  if ((kind == LBM_FLOW_POINT || kind == LBM_FLOW_PLANE || kind == LBM_FLOW_BOX) && !params)
    return fail(LBM_ERR_INVALID, "null flow parameters");
  if (kind == LBM_FLOW_PLANE && (params[0] < 0 || params[0] > 2))
    return fail(LBM_ERR_INVALID, "plane axis must be 0..2");
  if (kind == LBM_FLOW_MASK && !mask)
    return fail(LBM_ERR_INVALID, "null flow mask");
  FlowSpec fl{};
  fl.kind = kind;
  const int np = kind == LBM_FLOW_POINT ? 3 : (kind == LBM_FLOW_PLANE ? 2 : (kind == LBM_FLOW_BOX ? 6 : 0));
  for (int k = 0; k < np; ++k) fl.params[k] = params[k];
  if (induced)
    for (int i = 0; i < 27; ++i) fl.induced[i] = induced[i];
  if (kind == LBM_FLOW_MASK) {
    if (!c->flow_mask) {
      int rc = dev_alloc(c, (void**)&c->flow_mask, c->grid.n, "hipMalloc(flow mask)");
      if (rc) return rc;
    }
    int rc = h2d(c, c->flow_mask, mask, c->grid.n);
    if (rc) return rc;
    fl.mask = c->flow_mask;
  }
  c->flow = fl;
  return LBM_OK;
}

int lbm_stream(lbm_ctx* c) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_stream")) return rc;
  int rc = launch_ref_stream(c->grid, (const float*)c->f[c->cur],
                             (float*)c->f[c->cur ^ 1], c->stream);
  if (rc) return rc;
  c->cur ^= 1;
  return LBM_OK;
}

int lbm_collide(lbm_ctx* c, float tau) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_collide")) return rc;
  return launch_ref_collide(c->grid, (float*)c->f[c->cur], tau, nullptr,
                            c->stream);
}

int lbm_reflect(lbm_ctx* c, int with_force) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_reflect")) return rc;
  return reflect(c, with_force);
}

int lbm_flow(lbm_ctx* c) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_flow")) return rc;
  return launch_ref_flow(c->grid, (float*)c->f[c->cur], c->flow, c->stream);
}

int lbm_prime_points(lbm_ctx* c) { return check_ctx(c); }

int lbm_set_force(lbm_ctx* c, const float in[3]) {
  if (int rc = check_ctx(c)) return rc;
  if (!in) return fail(LBM_ERR_INVALID, "null force");
  return h2d(c, c->force, in, 3 * sizeof(float));
}

int lbm_get_force(lbm_ctx* c, float out[3]) {
  if (int rc = check_ctx(c)) return rc;
  if (!out) return fail(LBM_ERR_INVALID, "null force");
  return d2h(c, out, c->force, 3 * sizeof(float));
}

int lbm_step(lbm_ctx* c, int n) {
  if (int rc = check_ctx(c)) return rc;
  if (n < 0) return fail(LBM_ERR_INVALID, "negative step count");
  TraceRange tr("lbm_step");
  return c->cfg.mode == LBM_MODE_STANDARD ? step_standard(c, n)
                                          : step_reference_fused(c, n);
}

int lbm_step_route(const lbm_config* cfg, int n, int* kernel,
                   int32_t launches[LBM_MAX_LAUNCH_STEPS]) {
  if (int rc = validate_config(cfg)) return rc;
  if (cfg->mode != LBM_MODE_STANDARD)
    return fail(LBM_ERR_STATE, "lbm_step_route needs a standard-mode configuration");
  if (n < 0) return fail(LBM_ERR_INVALID, "negative step count");
  if (!kernel || !launches) return fail(LBM_ERR_INVALID, "null output");
  const StepPlan p =
      plan_steps(cfg->lattice, device_storage(cfg->mode, cfg->storage), make_grid(*cfg), n);
  *kernel = p.kernel;
  for (int k = 1; k <= LBM_MAX_LAUNCH_STEPS; ++k) launches[k - 1] = p.launches[k];
  return LBM_OK;
}

int lbm_step_each(lbm_ctx* const* ctxs, int32_t count, int n) {
  if (!ctxs || count < 0 || n < 0) return fail(LBM_ERR_INVALID, "bad arguments");
  TraceRange tr("lbm_step_each");
  for (int32_t k = 0; k < count; ++k) {
    if (int rc = check_ctx(ctxs[k])) return rc;
    if (ctxs[k]->cfg.mode != LBM_MODE_STANDARD)
      return fail(LBM_ERR_STATE, "lbm_step_each needs standard-mode lattices");
  }
  for (int s = 0; s < n; ++s)
    for (int32_t k = 0; k < count; ++k)
      if (int rc = step_standard(ctxs[k], 1)) return rc;
  return LBM_OK;
}

int lbm_step_reference(lbm_ctx* c, int n, int with_force) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = need_mode(c, LBM_MODE_REFERENCE, "lbm_step_reference")) return rc;
  if (n < 0) return fail(LBM_ERR_INVALID, "negative step count");
  TraceRange tr("lbm_step_reference");
  return step_reference_full(c, n, with_force);
}

int lbm_time_steps(lbm_ctx* c, int n, float* ms) {
  if (int rc = check_ctx(c)) return rc;
  if (!ms) return fail(LBM_ERR_INVALID, "null output");
  LBM_HIP(hipEventRecord(c->ev0, c->stream));
  int rc = api::lbm_step(c, n);
  if (rc) return rc;
  LBM_HIP(hipEventRecord(c->ev1, c->stream));
  LBM_HIP(hipEventSynchronize(c->ev1));
  LBM_HIP(hipEventElapsedTime(ms, c->ev0, c->ev1));
  return LBM_OK;
}

int lbm_time_steps_reference(lbm_ctx* c, int n, int with_force, float* ms) {
  if (int rc = check_ctx(c)) return rc;
  if (!ms) return fail(LBM_ERR_INVALID, "null output");
  int rc = rebuild_special(c);
  if (rc) return rc;
  LBM_HIP(hipEventRecord(c->ev0, c->stream));
  if ((rc = api::lbm_step_reference(c, n, with_force))) return rc;
  LBM_HIP(hipEventRecord(c->ev1, c->stream));
  LBM_HIP(hipEventSynchronize(c->ev1));
  LBM_HIP(hipEventElapsedTime(ms, c->ev0, c->ev1));
  return LBM_OK;
}

int lbm_moments(lbm_ctx* c, float* rho, float* u) {
  if (int rc = check_ctx(c)) return rc;
  const size_t N = c->grid.n;
  int rc;
  // rho and u staged in the context's buffer (4 N + 12 N bytes), kept
  // from call to call
  if (c->stage_bytes < 16 * N) {
    dev_free(c, &c->stage, c->stage_bytes);
    c->stage_bytes = 0;
    if ((rc = dev_alloc(c, &c->stage, 16 * N, "hipMalloc(moments staging)"))) return rc;
    c->stage_bytes = 16 * N;
  }
  return read_moments(c, c->stage, rho, u);
}

int lbm_conservation(lbm_ctx* c, double out[4]) {
  if (int rc = check_ctx(c)) return rc;
  if (!out) return fail(LBM_ERR_INVALID, "null output");
  int rc = launch_conservation(c->q, device_storage(c->cfg.mode, c->cfg.storage), c->grid, c->f[c->cur],
                               c->mask, c->red, c->red_cap, c->red_out,
                               c->stream);
  if (rc) return rc;
  return d2h(c, out, c->red_out, 4 * sizeof(double));
}

int lbm_test_coordinates(lbm_ctx* c, int* ok) {
  if (int rc = check_ctx(c)) return rc;
  if (!ok) return fail(LBM_ERR_INVALID, "null output");
  DevBuf counts, dok;
  int rc;
  if ((rc = counts.alloc(sizeof(uint32_t) * c->grid.n)) || (rc = dok.alloc(sizeof(int))))
    return rc;
  const int one = 1;
  LBM_HIP(hipMemsetAsync(counts.p, 0, sizeof(uint32_t) * c->grid.n, c->stream));
  if ((rc = h2d(c, dok.p, &one, sizeof(int)))) return rc;
  if ((rc = launch_test_coordinates(c->grid, (uint32_t*)counts.p, (int*)dok.p,
                                    c->stream)))
    return rc;
  return d2h(c, ok, dok.p, sizeof(int));
}

int lbm_measure_copy_bandwidth(int64_t bytes, int iters, double* gbs) {
  if (bytes < 16 || iters < 1 || !gbs)
    return fail(LBM_ERR_INVALID, "bad copy-bandwidth arguments");
  const uint64_t nbytes = (uint64_t)bytes / 16 * 16;
  DevBuf a, b;
  int rc;
  if ((rc = a.alloc(nbytes)) || (rc = b.alloc(nbytes))) return rc;
  hipStream_t s;
  LBM_HIP(hipStreamCreate(&s));
  hipEvent_t e0, e1;
  hipError_t e;
  if ((e = hipEventCreate(&e0)) != hipSuccess) {
    (void)hipStreamDestroy(s);
    return hip_fail(e, "hipEventCreate");
  }
  if ((e = hipEventCreate(&e1)) != hipSuccess) {
    (void)hipEventDestroy(e0);
    (void)hipStreamDestroy(s);
    return hip_fail(e, "hipEventCreate");
  }
  float ms = 0.0f;
  rc = LBM_OK;
  if ((e = hipMemsetAsync(a.p, 0, nbytes, s)) != hipSuccess) rc = hip_fail(e, "hipMemsetAsync");
  for (int w = 0; w < 3 && rc == LBM_OK; ++w) rc = launch_copy_stream(a.p, b.p, nbytes, s);
  if (rc == LBM_OK && (e = hipEventRecord(e0, s)) != hipSuccess) rc = hip_fail(e, "hipEventRecord");
  for (int k = 0; k < iters && rc == LBM_OK; ++k) rc = launch_copy_stream(a.p, b.p, nbytes, s);
  if (rc == LBM_OK && (e = hipEventRecord(e1, s)) != hipSuccess) rc = hip_fail(e, "hipEventRecord");
  if (rc == LBM_OK && (e = hipEventSynchronize(e1)) != hipSuccess) rc = hip_fail(e, "hipEventSynchronize");
  if (rc == LBM_OK && (e = hipEventElapsedTime(&ms, e0, e1)) != hipSuccess) rc = hip_fail(e, "hipEventElapsedTime");
  (void)hipStreamSynchronize(s);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipStreamDestroy(s);
  if (rc == LBM_OK) *gbs = 2.0 * (double)nbytes * iters / (ms * 1e-3) / 1e9;
  return rc;
}

int64_t lbm_random_spheres(int32_t nx, int32_t ny, int32_t nz, uint64_t seed,
                           double frac, double rmin, double rmax,
                           int32_t periodic_x, uint8_t* solid,
                           int64_t max_spheres, double* spheres) {
#pragma clang fp contract(off)
  if (nx < 1 || ny < 1 || nz < 1 || !solid || !(frac >= 0.0 && frac <= 1.0) ||
      !(rmin > 0.0) || rmax < rmin) {
    set_error("bad random-sphere arguments");
    return -LBM_ERR_INVALID;
  }
  const int64_t N = (int64_t)nx * ny * nz;
  std::memset(solid, 0, (size_t)N);
  std::mt19937_64 gen(seed);
  auto u01 = [&gen]() { return (double)(gen() >> 11) * 0x1.0p-53; };
  int64_t count = 0, ns = 0;
  const double target = frac * (double)N;
  while ((double)count < target) {
    const double c[3] = {u01() * nx, u01() * ny, u01() * nz};
    const double r = rmin + (rmax - rmin) * u01();
    if (spheres && ns < max_spheres) {
      spheres[4 * ns + 0] = c[0];
      spheres[4 * ns + 1] = c[1];
      spheres[4 * ns + 2] = c[2];
      spheres[4 * ns + 3] = r;
    }
    ++ns;
    const int64_t lo[3] = {(int64_t)std::floor(c[0] - r), (int64_t)std::floor(c[1] - r),
                           (int64_t)std::floor(c[2] - r)};
    const int64_t hi[3] = {(int64_t)std::ceil(c[0] + r), (int64_t)std::ceil(c[1] + r),
                           (int64_t)std::ceil(c[2] + r)};
    const double r2 = r * r;
    for (int64_t x = lo[0]; x <= hi[0]; ++x) {
      int64_t xi = x;
      if (xi < 0 || xi >= nx) {
        if (!periodic_x) continue;
        xi = ((xi % nx) + nx) % nx;
      }
      const double dx = (double)x - c[0];
      const double dx2 = dx * dx;
      for (int64_t y = std::max<int64_t>(lo[1], 0); y <= hi[1] && y < ny; ++y) {
        const double dy = (double)y - c[1];
        const double dxy = dx2 + dy * dy;
        for (int64_t z = std::max<int64_t>(lo[2], 0); z <= hi[2] && z < nz; ++z) {
          const double dz = (double)z - c[2];
          if (dxy + dz * dz <= r2) {
            uint8_t& s = solid[z + nz * (y + ny * xi)];
            if (!s) {
              s = 1;
              ++count;
            }
          }
        }
      }
    }
  }
  return ns;
}

}  // namespace api
}  // namespace lbm
