// Tables of the reference mode's geometry, built on the GPU from the flag
// bytes and the reflection records: the list of flagged nodes (staged
// reflection pass) and the receiver tables of the fused step.
//
// Every slot s (1..80) of a reflecting node x with direction d (1..26) whose
// target t = x + e_d lies in the box is an entry of group (t, d).  All
// entries of a group come from the one node x = t - e_d, so a record's
// groups are the directions that occur among its slots: each record is
// handled by itself, and prefix sums over the records (in node order) and
// over the receivers place what it writes.
//   - The gather's threads take the groups by reflecting node, then
//     direction; gsrc, gbeg, gid and the entries (eidx, ew, es: a group's
//     slots in ascending s, the order in which the staged pass adds them)
//     follow that order.
//   - gid is a group's slot of gsum: receivers in node order, then
//     direction (rxbase[t] + the directions below d that arrive at t).
// Targets must not be flagged: the staged pass would otherwise race between
// adding to a target and zeroing it.
//
// Built on the host these tables took 23 ms for 14,683 records on 96^3 (1 ms
// on 33 x 32 x 31); uploading the records and building them here takes 0.9
// ms, 0.25 of it kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "lbm_internal.h"
#include "lbm_lattice.h"
#include "lbm_layout.h"
#include "lbm_scan.h"

namespace lbm {
namespace {

using L27 = Lat<27>;
constexpr int kBlock = 256;
constexpr uint32_t kNone = ~0u;

// Read back once: table sizes, and what is wrong with the geometry (kNone /
// ~0: nothing).
struct Totals {
  uint32_t special, active, groups, entries;
  uint32_t dup;        // first record of a node that has one already
  uint32_t outside;    // first reflecting node with a record that is not internal
  unsigned long long target;  // node << 7 | slot of the first flagged target
};

// A direction's slots: 5 bits each, six to a word.
__device__ __forceinline__ int slot_dir(const uint32_t* __restrict__ words, int s) {
  return (int)((words[s / 6] >> (5 * (s % 6))) & 0x1Fu);
}

__device__ __forceinline__ void place(const Grid& g, uint32_t n, int& x, int& y, int& z) {
  const uint32_t t = g.dz.div(n);
  z = (int)(n - t * g.nz);
  x = (int)g.dy.div(t);
  y = (int)(t - (uint32_t)x * g.ny);
}

// Whether (x, y, z) + sign e_d lies in the box, and its node.
__device__ __forceinline__ bool neighbour(const Grid& g, int x, int y, int z, int d, int sign,
                                          uint32_t& n) {
  const int a = x + sign * L27::E[d][0], b = y + sign * L27::E[d][1], c = z + sign * L27::E[d][2];
  n = (uint32_t)c + g.nz * ((uint32_t)b + g.ny * (uint32_t)a);
  return a >= 0 && b >= 0 && c >= 0 && a < (int)g.nx && b < (int)g.ny && c < (int)g.nz;
}

__global__ void __launch_bounds__(kBlock)
    k_rx_clear(uint32_t* __restrict__ rec_of, uint32_t n, Totals* __restrict__ tot) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) rec_of[i] = kNone;
  if (i == 0) {
    *tot = Totals{};
    tot->dup = tot->outside = kNone;
    tot->target = ~0ull;
  }
}

// rec_of[node] = its first record
__global__ void __launch_bounds__(kBlock)
    k_rx_rec_of(const int32_t* __restrict__ node, uint32_t nrec, uint32_t* __restrict__ rec_of) {
  const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
  if (r < nrec) atomicMin(&rec_of[node[r]], r);
}

__global__ void __launch_bounds__(kBlock)
    k_rx_check(const int32_t* __restrict__ node, uint32_t nrec,
               const uint32_t* __restrict__ rec_of, const uint8_t* __restrict__ flags,
               Totals* __restrict__ tot) {
  const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= nrec) return;
  const uint32_t n = (uint32_t)node[r];
  if (rec_of[n] != r) atomicMin(&tot->dup, r);
  if ((flags[n] & (LBM_FLAG_REFLECTED | LBM_FLAG_INTERNAL)) == LBM_FLAG_REFLECTED)
    atomicMin(&tot->outside, n);
}

struct SpecialIn {
  const uint8_t* flags;
  __device__ uint32_t operator()(uint32_t n) const { return flags[n] ? 1u : 0u; }
};
struct SpecialOut {
  int32_t* special;
  int32_t* rec;
  const uint32_t* rec_of;  // null without records
  __device__ void operator()(uint32_t n, uint32_t v, uint32_t at) const {
    if (!v) return;
    special[at] = (int32_t)n;
    rec[at] = rec_of ? (int32_t)rec_of[n] : -1;
  }
};
// reflecting nodes that have a record
struct ActiveIn {
  const uint8_t* flags;
  const uint32_t* rec_of;
  __device__ uint32_t operator()(uint32_t n) const {
    return (flags[n] & LBM_FLAG_REFLECTED) && rec_of[n] != kNone ? 1u : 0u;
  }
};
struct ActiveOut {
  uint32_t* node;
  uint32_t* rec;
  const uint32_t* rec_of;
  __device__ void operator()(uint32_t n, uint32_t v, uint32_t at) const {
    if (!v) return;
    node[at] = n;
    rec[at] = rec_of[n];
  }
};

// Groups (as a mask of directions) and entries of every active record.
__global__ void __launch_bounds__(kBlock)
    k_rx_count(Grid g, const Totals* __restrict__ tot_in, const uint32_t* __restrict__ act_node,
               const uint32_t* __restrict__ act_rec, const uint32_t* __restrict__ dirs,
               const uint8_t* __restrict__ flags, uint32_t* __restrict__ gmask,
               uint32_t* __restrict__ ecount, Totals* __restrict__ tot) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= tot_in->active) return;
  const uint32_t n = act_node[i];
  const uint32_t* words = dirs + 14 * (size_t)act_rec[i];
  int x, y, z;
  place(g, n, x, y, z);
  uint32_t mask = 0, count = 0;
  for (int s = 1; s < 81; ++s) {
    const int d = slot_dir(words, s);
    uint32_t t;
    if (d == 0 || d > 26 || !neighbour(g, x, y, z, d, 1, t)) continue;
    if (flags[t]) atomicMin(&tot->target, (unsigned long long)n << 7 | (unsigned)s);
    mask |= 1u << d;
    ++count;
  }
  gmask[i] = mask;
  ecount[i] = count;
}

struct GroupsIn {
  const uint32_t* gmask;
  const Totals* tot;
  __device__ uint32_t operator()(uint32_t i) const {
    return i < tot->active ? (uint32_t)__popc(gmask[i]) : 0u;
  }
};
struct EntriesIn {
  const uint32_t* ecount;
  const Totals* tot;
  __device__ uint32_t operator()(uint32_t i) const { return i < tot->active ? ecount[i] : 0u; }
};
struct Offsets {
  uint32_t* to;
  __device__ void operator()(uint32_t i, uint32_t, uint32_t at) const { to[i] = at; }
};

// The directions that arrive at every receiver (lane d: direction d), and
// the tiles whose nodes the next step's gather and fused pass read (lane =
// column of nodes): those within two nodes of a reflecting node (the gather
// reads those within one, and the fused pass all of them; on the 128^3
// angled cube a reach of 2 to 8 nodes gave 85.0-85.1 us per step, 1 node
// 85.6, 16 nodes 85.6-85.7: the caches start to lose them).  One wavefront
// per active record.
__global__ void __launch_bounds__(kBlock)
    k_rx_mark(Grid g, uint32_t nactive, const uint32_t* __restrict__ act_node,
              const uint32_t* __restrict__ gmask, uint32_t* __restrict__ inmask,
              uint8_t* __restrict__ near) {
  constexpr int kReach = 2, kSide = 2 * kReach + 1;
  const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (i >= nactive) return;
  const int lane = threadIdx.x & 63;
  int x, y, z;
  place(g, act_node[i], x, y, z);
  uint32_t t;
  if (lane < 27 && ((gmask[i] >> lane) & 1u) && neighbour(g, x, y, z, lane, 1, t))
    atomicOr(&inmask[t], 1u << lane);
  const int a = x + lane / kSide - kReach, b = y + lane % kSide - kReach;
  if (lane >= kSide * kSide || a < 0 || b < 0 || a >= (int)g.nx || b >= (int)g.ny) return;
  const uint32_t row = g.nz * ((uint32_t)b + g.ny * (uint32_t)a);
  const uint32_t z0 = (uint32_t)max(z - kReach, 0), z1 = (uint32_t)min(z + kReach, (int)g.nz - 1);
  // a byte per tile, which every thread sets to the same (bits of shared
  // words took 0.5 ms of contended atomics for 14,683 records)
  for (t = (row + z0) / kTile; t <= (row + z1) / kTile; ++t) near[t] = 1;
}

// 2-bit classes: 0 plain, 1 receiver, 2 internal; a bit for each near tile.
__global__ void __launch_bounds__(kBlock)
    k_rx_class(uint32_t n, const uint8_t* __restrict__ flags, const uint32_t* __restrict__ inmask,
               const uint8_t* __restrict__ near, uint32_t* __restrict__ cls,
               uint32_t* __restrict__ keep) {
  const uint32_t w = blockIdx.x * kBlock + threadIdx.x;
  if (w >= (n + 15) / 16) return;
  const uint32_t tiles = (n + kTile - 1) / kTile;
  if (w < (tiles + 31) / 32) {
    uint32_t bits = 0;
    for (uint32_t k = 0; k < 32 && w * 32 + k < tiles; ++k) bits |= (uint32_t)near[w * 32 + k] << k;
    keep[w] = bits;
  }
  uint32_t out = 0;
  for (uint32_t k = 0; k < 16 && w * 16 + k < n; ++k) {
    const uint32_t i = w * 16 + k;
    const uint32_t c = (flags[i] & LBM_FLAG_INTERNAL) ? 2u : (inmask[i] ? 1u : 0u);
    out |= c << (2 * k);
  }
  cls[w] = out;
}

struct InmaskIn {
  const uint32_t* inmask;
  __device__ uint32_t operator()(uint32_t n) const { return (uint32_t)__popc(inmask[n]); }
};
struct RxBaseOut {
  int32_t* rxbase;
  __device__ void operator()(uint32_t n, uint32_t v, uint32_t at) const {
    rxbase[n] = v ? (int32_t)at : -1;
  }
};

// One wavefront per active record, lane d its direction d.
__global__ void __launch_bounds__(kBlock)
    k_rx_fill(Grid g, uint32_t nactive, const uint32_t* __restrict__ act_node,
              const uint32_t* __restrict__ act_rec, const uint32_t* __restrict__ dirs,
              const float* __restrict__ weights, const uint32_t* __restrict__ gmask,
              const uint32_t* __restrict__ goff, const uint32_t* __restrict__ eoff,
              const uint32_t* __restrict__ inmask, const int32_t* __restrict__ rxbase,
              uint32_t* __restrict__ gsrc, uint32_t* __restrict__ gbeg,
              uint32_t* __restrict__ gid, uint32_t* __restrict__ eidx, float* __restrict__ ew,
              uint8_t* __restrict__ es) {
  const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (i >= nactive) return;
  const int d = threadIdx.x & 63;
  const uint32_t n = act_node[i], mask = gmask[i];
  const uint32_t* words = dirs + 14 * (size_t)act_rec[i];
  const float* w = weights + 81 * (size_t)act_rec[i];
  int x, y, z;
  place(g, n, x, y, z);
  const bool mine = d < 27 && ((mask >> d) & 1u);
  uint32_t count = 0;
  if (mine)
    for (int s = 1; s < 81; ++s) count += slot_dir(words, s) == d ? 1u : 0u;
  uint32_t inc = count;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const uint32_t up = __shfl_up(inc, o, 64);
    if (d >= o) inc += up;
  }
  if (!mine) return;
  uint32_t at = eoff[i] + inc - count;
  const uint32_t gi = goff[i] + (uint32_t)__popc(mask & ((1u << d) - 1u));
  uint32_t t;
  (void)neighbour(g, x, y, z, d, 1, t);
  gsrc[gi] = pidx<27>(n, d);
  gbeg[gi] = at;
  gid[gi] = (uint32_t)rxbase[t] + (uint32_t)__popc(inmask[t] & ((1u << d) - 1u));
  for (int s = 1; s < 81; ++s) {
    if (slot_dir(words, s) != d) continue;
    // the streamed value of direction k that slot s reflects: A_k(x - e_k),
    // 0 outside
    const int k = s / 3;
    uint32_t src;
    eidx[at] = neighbour(g, x, y, z, k, -1, src) ? pidx<27>(src, k) : kNone;
    ew[at] = w[s];
    es[at] = (uint8_t)s;
    ++at;
  }
}

inline unsigned blocks_for(uint64_t n) { return (unsigned)std::max<uint64_t>((n + kBlock - 1) / kBlock, 1); }

int fail_geometry(const lbm_ctx* c, const Totals& t, const int32_t* rec_node_dev) {
  if (t.dup != kNone) {
    int32_t node = -1;
    LBM_HIP(hipMemcpy(&node, rec_node_dev + t.dup, sizeof node, hipMemcpyDeviceToHost));
    return fail(LBM_ERR_INVALID, "two reflection records for node " + std::to_string(node));
  }
  if (t.outside != kNone)
    return fail(LBM_ERR_INVALID, "reflecting node " + std::to_string(t.outside) +
                                     " is not internal (reflection runs in place and needs "
                                     "reflecting nodes inside the obstacle)");
  // the target of the first flagged link, from its node and slot
  const uint32_t n = (uint32_t)(t.target >> 7), s = (uint32_t)(t.target & 127u);
  int32_t rec = -1;
  uint32_t word = 0;
  std::vector<int32_t> nodes((size_t)c->nrec);
  LBM_HIP(hipMemcpy(nodes.data(), rec_node_dev, sizeof(int32_t) * nodes.size(), hipMemcpyDeviceToHost));
  for (size_t r = 0; r < nodes.size() && rec < 0; ++r)
    if ((uint32_t)nodes[r] == n) rec = (int32_t)r;
  LBM_HIP(hipMemcpy(&word, c->rec_dirs + 14 * (size_t)rec + s / 6, sizeof word, hipMemcpyDeviceToHost));
  const int d = (int)((word >> (5 * (s % 6))) & 0x1Fu);
  const Grid& g = c->grid;
  const int64_t target = (int64_t)n + L27::E[d][2] +
                         (int64_t)g.nz * (L27::E[d][1] + (int64_t)g.ny * L27::E[d][0]);
  return fail(LBM_ERR_INVALID, "reflection target " + std::to_string(target) +
                                   " is a flagged node (targets must be fluid)");
}

}  // namespace

int build_receivers(lbm_ctx* c) {
  const Grid& g = c->grid;
  const uint32_t N = g.n, nrec = (uint32_t)c->nrec;
  const hipStream_t s = c->stream;
  c->nspecial = 0;
  c->ref_geom = false;
  c->ref_ngrp = c->ref_nent = 0;
  DevArena tmp;
  const size_t o_tot = tmp.add(sizeof(Totals));
  const size_t o_rec = tmp.add(4ull * N);
  const size_t o_node = tmp.add(4ull * nrec), o_arec = tmp.add(4ull * nrec);
  const size_t o_gm = tmp.add(4ull * nrec), o_ec = tmp.add(4ull * nrec);
  const size_t o_go = tmp.add(4ull * nrec), o_eo = tmp.add(4ull * nrec);
  const size_t tiles_n = 4ull * (scan_tiles(N) + 1), tiles_r = 4ull * (scan_tiles(nrec) + 1);
  const size_t o_s1 = tmp.add(tiles_n), o_s2 = tmp.add(tiles_n), o_s3 = tmp.add(tiles_r),
               o_s4 = tmp.add(tiles_r);
  const size_t o_near = tmp.add((N + kTile - 1) / kTile);
  int rc;
  if ((rc = tmp.alloc("hipMalloc(receiver tables)"))) return rc;
  Totals* tot = tmp.at<Totals>(o_tot);
  uint32_t* rec_of = tmp.at<uint32_t>(o_rec);
  uint32_t *act_node = tmp.at<uint32_t>(o_node), *act_rec = tmp.at<uint32_t>(o_arec);
  uint32_t *gmask = tmp.at<uint32_t>(o_gm), *ecount = tmp.at<uint32_t>(o_ec);
  uint32_t *goff = tmp.at<uint32_t>(o_go), *eoff = tmp.at<uint32_t>(o_eo);
  hipLaunchKernelGGL(k_rx_clear, dim3(blocks_for(N)), dim3(kBlock), 0, s, rec_of, N, tot);
  const SpecialIn special_in{c->flags};
  if ((rc = launch_scan_sums(special_in, N, tmp.at<uint32_t>(o_s1), &tot->special, s))) return rc;
  if (nrec) {
    hipLaunchKernelGGL(k_rx_rec_of, dim3(blocks_for(nrec)), dim3(kBlock), 0, s, c->rec_node, nrec,
                       rec_of);
    hipLaunchKernelGGL(k_rx_check, dim3(blocks_for(nrec)), dim3(kBlock), 0, s, c->rec_node, nrec,
                       rec_of, c->flags, tot);
    const ActiveIn active{c->flags, rec_of};
    if ((rc = launch_scan_sums(active, N, tmp.at<uint32_t>(o_s2), &tot->active, s)) ||
        (rc = launch_scan_write(active, N, tmp.at<uint32_t>(o_s2),
                                ActiveOut{act_node, act_rec, rec_of}, s)))
      return rc;
    hipLaunchKernelGGL(k_rx_count, dim3(blocks_for(nrec)), dim3(kBlock), 0, s, g, tot, act_node,
                       act_rec, c->rec_dirs, c->flags, gmask, ecount, tot);
    const GroupsIn groups{gmask, tot};
    const EntriesIn entries{ecount, tot};
    if ((rc = launch_scan_sums(groups, nrec, tmp.at<uint32_t>(o_s3), &tot->groups, s)) ||
        (rc = launch_scan_write(groups, nrec, tmp.at<uint32_t>(o_s3), Offsets{goff}, s)) ||
        (rc = launch_scan_sums(entries, nrec, tmp.at<uint32_t>(o_s4), &tot->entries, s)) ||
        (rc = launch_scan_write(entries, nrec, tmp.at<uint32_t>(o_s4), Offsets{eoff}, s)))
      return rc;
  }
  LBM_HIP(hipGetLastError());
  Totals t{};
  LBM_HIP(hipMemcpyAsync(&t, tot, sizeof t, hipMemcpyDeviceToHost, s));
  LBM_HIP(hipStreamSynchronize(s));
  if (t.dup != kNone || t.outside != kNone || t.target != ~0ull) return fail_geometry(c, t, c->rec_node);
  if (t.entries >= 1u << 31) return fail(LBM_ERR_UNSUPPORTED, "too many reflected links");

  // the tables, in one allocation that the context keeps and reuses
  const uint32_t words = (N + 15) / 16, kwords = (N + 64 * 32 - 1) / (64 * 32);
  const bool geom = t.special > 0;
  const int npart = ref_gather_partials(t.groups);
  const int fblocks = std::max(1, ref_reflect_blocks((int32_t)t.special));
  DevArena lay;  // offsets only
  const size_t p_sp = lay.add(4ull * t.special), p_sr = lay.add(4ull * t.special);
  const size_t p_fp = lay.add(12ull * fblocks);
  const size_t p_cls = lay.add(geom ? 4ull * words : 0);
  const size_t p_in = lay.add(geom ? 4ull * N : 0), p_keep = lay.add(geom ? 4ull * kwords : 0);
  const size_t p_rx = lay.add(geom ? 4ull * N : 0);
  const size_t p_gsrc = lay.add(4ull * t.groups), p_gbeg = lay.add(4ull * t.groups);
  const size_t p_gid = lay.add(4ull * t.groups), p_gsum = lay.add(4ull * t.groups);
  const size_t p_ei = lay.add(4ull * t.entries), p_ew = lay.add(4ull * t.entries);
  const size_t p_es = lay.add(t.entries);
  const size_t p_part = lay.add(12ull * std::max(npart, 1));
  if (c->ref_tables_bytes < lay.bytes || c->ref_tables_bytes / 4 > lay.bytes) {
    if (c->ref_tables) {
      (void)hipFree(c->ref_tables);
      c->device_bytes -= (int64_t)c->ref_tables_bytes;
    }
    c->ref_tables = nullptr;
    c->ref_tables_bytes = 0;
    const hipError_t e = hipMalloc(&c->ref_tables, lay.bytes);
    if (e != hipSuccess) {
      c->ref_tables = nullptr;
      return hip_fail(e, "hipMalloc(receiver tables)");
    }
    c->ref_tables_bytes = lay.bytes;
    c->device_bytes += (int64_t)lay.bytes;
  }
  char* base = (char*)c->ref_tables;
  c->special = (int32_t*)(base + p_sp);
  c->special_rec = (int32_t*)(base + p_sr);
  c->force_partials = (float*)(base + p_fp);
  c->ref_cls = (uint32_t*)(base + p_cls);
  c->ref_inmask = (uint32_t*)(base + p_in);
  c->ref_keep = (uint32_t*)(base + p_keep);
  c->ref_rxbase = (int32_t*)(base + p_rx);
  c->ref_gsrc = (uint32_t*)(base + p_gsrc);
  c->ref_gbeg = (uint32_t*)(base + p_gbeg);
  c->ref_gid = (uint32_t*)(base + p_gid);
  c->ref_gsum = (float*)(base + p_gsum);
  c->ref_eidx = (uint32_t*)(base + p_ei);
  c->ref_ew = (float*)(base + p_ew);
  c->ref_es = (uint8_t*)(base + p_es);
  c->ref_partials = (float*)(base + p_part);
  if (geom) {
    if ((rc = launch_scan_write(special_in, N, tmp.at<uint32_t>(o_s1),
                                SpecialOut{c->special, c->special_rec, nrec ? rec_of : nullptr}, s)))
      return rc;
    uint8_t* near = tmp.at<uint8_t>(o_near);
    LBM_HIP(hipMemsetAsync(c->ref_inmask, 0, 4ull * N, s));
    LBM_HIP(hipMemsetAsync(near, 0, (N + kTile - 1) / kTile, s));
    if (t.active)
      hipLaunchKernelGGL(k_rx_mark, dim3((t.active + kBlock / 64 - 1) / (kBlock / 64)), dim3(kBlock),
                         0, s, g, t.active, act_node, gmask, c->ref_inmask, near);
    hipLaunchKernelGGL(k_rx_class, dim3(blocks_for(words)), dim3(kBlock), 0, s, N, c->flags,
                       c->ref_inmask, near, c->ref_cls, c->ref_keep);
    const InmaskIn in{c->ref_inmask};
    if ((rc = launch_scan_sums(in, N, tmp.at<uint32_t>(o_s2), &tot->groups, s)) ||
        (rc = launch_scan_write(in, N, tmp.at<uint32_t>(o_s2), RxBaseOut{c->ref_rxbase}, s)))
      return rc;
    if (t.active)
      hipLaunchKernelGGL(k_rx_fill, dim3((t.active + kBlock / 64 - 1) / (kBlock / 64)), dim3(kBlock),
                         0, s, g, t.active, act_node, act_rec, c->rec_dirs, c->rec_w, gmask, goff,
                         eoff, c->ref_inmask, c->ref_rxbase, c->ref_gsrc, c->ref_gbeg, c->ref_gid,
                         c->ref_eidx, c->ref_ew, c->ref_es);
    LBM_HIP(hipGetLastError());
  }
  LBM_HIP(hipStreamSynchronize(s));  // the working arrays go
  c->nspecial = (int32_t)t.special;
  c->ref_geom = geom;
  c->ref_ngrp = t.groups;
  c->ref_nent = t.entries;
  return LBM_OK;
}

}  // namespace lbm
