// Several steps of a D2Q9 lattice in one pass over memory.
//
// A wavefront takes a strip of 64 consecutive y (one node per lane) and
// walks it along x, row by row.  Each row of populations is read once; K
// stages in registers then apply K steps, stage s (1..K) one row behind
// stage s - 1: when row X + 1 after s - 1 steps is there, row X after s
// steps can be formed, since a D2Q9 update needs the rows X - 1, X and
// X + 1 only.  After the last stage the row is written: the populations are
// read and written once for K steps, instead of K times.
//
// Neighbours along y sit in the neighbouring lanes (one DPP lane shift per
// direction that has a y component), so there is no LDS, no barrier and,
// but for the row's own address, no index arithmetic.  What it costs: the
// outermost K lanes at a strip's inner ends and the K - 1 rows beside a
// chunk's ends are computed by both neighbours (56 of 64 lanes store).
// Lattices narrower than a wavefront put several x-chunks side by side in
// one.
//
// One step at a time is bound by HBM (FP32, FP64) or by HBM and vector
// instructions alike (16 bits); four steps a pass are bound by vector
// instructions: 100-150 a node and step, of which the collision is 90
// (115 with a body force).  Measured per step on MI355X, one step at a time
// against this: 4096^2 FP32 204 -> 92.6 us, FP64 404 -> 168, FP16 channel
// 104 -> 90 and cavity 102 -> 70.6; 256 lattices of 32 to 512 a side (6.7 M
// nodes) FP32 81.8 -> 43.4, FP64 161 -> 76, FP16 55 -> 45.5.  Two nodes per
// lane halve the lane shifts but double the registers: 2 wavefronts per
// SIMD, 111 us against 102 for 4096^2 FP32.  Non-temporal stores cost 25 %
// (a strip's ends share cache lines with the next strip's, which meet in L2
// otherwise).
//
// The per-node arithmetic is std_collide_node on the same inputs, rounded
// to the stored type between stages, so K steps give the same bytes as K
// single steps.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "lbm_step_node.h"

namespace lbm {

constexpr uint32_t kSweepHalo = 4;  // lanes kept beside a strip: the largest K

// How a lattice is cut for the sweep (sweep_plan, on the host).
struct SweepPlan {
  uint32_t strips;   // strips along y
  uint32_t stride;   // output nodes of a strip (walled: of an inner one)
  uint32_t group;    // lanes of one x-chunk: 64, or fewer where several fit
  uint32_t groups;   // x-chunks side by side in a wavefront
  uint32_t rows;     // rows of an x-chunk, even
  uint32_t units;    // wavefronts of the whole lattice
};

// Strips along y of a lattice.
inline uint32_t sweep_strips(const Grid& g) {
  constexpr uint32_t H = kSweepHalo, W = 64 - 2 * H;
  if (g.flags & kWrapY) return g.ny + 2 * H <= 64 ? 1 : (g.ny + W - 1) / W;
  return g.ny <= 64 ? 1 : (g.ny - 2 * H + W - 1) / W;
}

// rows: wanted rows per x-chunk.
inline SweepPlan sweep_plan(const Grid& g, uint32_t rows) {
  SweepPlan p{};
  constexpr uint32_t H = kSweepHalo;
  const bool per = (g.flags & kWrapY) != 0;
  const uint32_t whole = per ? g.ny + 2 * H : g.ny;  // lanes of all of a row
  p.group = 64;
  p.groups = 1;
  p.strips = sweep_strips(g);
  if (whole <= 64) {
    p.stride = g.ny;
    p.group = whole;
    p.groups = 64 / whole;
  } else {
    p.stride = 64 - 2 * H;
  }
  rows = rows < 1 ? 1 : (rows > g.nx ? g.nx : rows);
  uint32_t chunks = (g.nx + rows - 1) / rows;
  p.groups = p.groups > chunks ? chunks : p.groups;
  // whole groups of chunks, then rows spread evenly over them
  chunks = (chunks + p.groups - 1) / p.groups * p.groups;
  p.rows = ((g.nx + chunks - 1) / chunks + 1) / 2 * 2;
  chunks = (g.nx + p.rows - 1) / p.rows;
  p.units = p.strips * ((chunks + p.groups - 1) / p.groups);
  return p;
}

// Wavefronts of a sweep that fit the GPU together: 256 CUs x 4 SIMDs x 3
// (2 with FP64 storage: the stages' registers).
inline uint32_t sweep_slots(int storage) { return storage == LBM_STORE_F64 ? 2048u : 3072u; }

// Rows per x-chunk for a pass over some lattices (count of them, grid(i)
// gives one): the fewest with which every slot gets one chunk, or, where
// that takes more than 64 rows, that many chunks one after another.  A chunk
// of r rows computes r + K - 1, so short ones waste work; but more chunks
// than whole rounds of the slots leave most slots idle in the last round
// (4096^2 FP32, K = 4: 98 or 49 rows, one round or two, 90-93 us per step;
// 73 rows, 1.35 rounds, 100 us).
constexpr uint64_t kSweepLooks = 16384;
template <class GridOf>
uint32_t sweep_chunk_rows(size_t count, GridOf&& grid, int storage) {
  const uint64_t slots = sweep_slots(storage);
  uint64_t strip_rows = 0;
  uint32_t longest = 1;
  for (size_t i = 0; i < count; ++i) {
    const Grid& g = grid(i);
    strip_rows += (uint64_t)sweep_strips(g) * g.nx;
    longest = g.nx > longest ? g.nx : longest;
  }
  const uint64_t one = (strip_rows + slots - 1) / slots;  // rows of one round
  const uint64_t rounds = one > 64 ? (one + 63) / 64 : 1;
  uint32_t rows = (uint32_t)((one + rounds - 1) / rounds);
  rows = rows < 4 ? 4 : (rows + 1) / 2 * 2;
  auto units_at = [&](uint32_t r) {
    uint64_t units = 0;
    for (size_t i = 0; i < count; ++i) units += sweep_plan(grid(i), r).units;
    return units;
  };
  // where the lattices are more than the slots, no length makes them fit
  if (rows < longest && units_at(longest) > rounds * slots)
    return rows + (longest - rows + 1) / 2 * 2;
  // Row by row as long as that is quick, then in growing steps: this runs
  // whenever a member comes or goes (3,500 lattices of 16^2 and one of 4000 x
  // 64 took 48 ms row by row).
  uint32_t step = 2;
  for (uint64_t looked = 0; rows < longest; rows += step) {
    if (units_at(rows) <= rounds * slots) break;
    looked += count;
    if (looked > kSweepLooks) step = (rows / 2 + 1) / 2 * 2;
  }
  return rows;
}

// Smallest FP32 / FP64 lattice that a single-lattice sweep is used for (the
// lattices below are stepped in boxes, except those too narrow for them:
// 512^2 FP32 one step at a time 6.48, in sweeps 4.6-5.0, in boxes 3.0 us per
// step); a smaller one has too few wavefronts, which walk too many rows one
// after another.
constexpr uint32_t kSweepMinNodes = 200000;

// Whether a lattice's rows are long enough, and enough of them, for a sweep;
// nodes: of all that are swept together.  Several chunks of short rows share
// a wavefront, whose loads and stores then scatter: per step against one at a
// time, FP32 rows of 1 / 2 / 4 / 8 / 16 nodes 6 M nodes 5.6 / 3.2 / 1.4 / 0.79
// / 0.51, 1 M nodes 6.2 / 3.0 / 1.4 / 1.4 / 0.83; FP64 6 M 3.0 / 1.5 / 0.82 /
// 0.49 / 0.38, 1 M 3.8 / 1.7 / 1.4 / 1.4 / 0.79; FP16 9 M rows of 8 / 16 / 24
// 1.4 / 0.9-1.1 / 0.85.  A chunk of few rows is mostly rim: a single row FP32
// 6 M 1.35, two 0.74; FP16 9 M 2 / 4 / 8 rows 1.4-1.6 / 0.97-1.1 / 0.8.
inline bool sweep_fits(const Grid& g, int storage, uint64_t nodes) {
  const size_t bytes = storage_bytes(storage);
  if (bytes == 2) return g.nx >= 8 && g.ny >= 24;
  const uint32_t row = nodes >= 4000000 && bytes == 8 ? 4 : nodes >= 2000000 ? 8 : 16;
  return g.nx >= 2 && g.ny >= row;
}

// What a launch of k steps costs ([k], k of 1 to 4), in any unit.
struct StepCosts {
  double of[5];
};
// Sweeps, in single steps (medians over 0.2 to 17 M nodes): two steps a pass
// save little, with 16 bits nothing, so a call of 4 goes by 3 and 1 (4096^2
// FP16 channel 449 -> 390 us; by twos it was slower than by ones).
inline StepCosts sweep_costs(int storage) {
  switch (storage_bytes(storage)) {
    case 2: return {{0.0, 1.0, 2.05, 2.25, 2.9}};
    case 8: return {{0.0, 1.0, 1.45, 1.5, 1.8}};
    default: return {{0.0, 1.0, 1.6, 1.75, 2.2}};
  }
}

// Splits n steps into launches of 1 to 4 (launches[k]: how many of k steps) at
// the least cost.  As many launches, odd or even, as there are steps, so that
// the current buffer is the one after single steps: those of 2 and 4 are even
// in number together.
inline void split_steps(int n, const StepCosts& c, int* launches) {
  const int most = c.of[4] < 4 * c.of[1] ? 4 : 1;
  if (n > 24) {  // the bulk of a long call
    const int eights = (n - 16) / 8;
    launches[most] += 8 / most * eights;
    n -= 8 * eights;
  }
  double best = 0.0;
  int take[5] = {0, -1, 0, 0, 0};
  for (int f = n / 4; f >= 0; --f)
    for (int t = (n - 4 * f) / 3; t >= 0; --t)
      for (int w = (n - 4 * f - 3 * t) / 2; w >= 0; --w) {
        if ((f + w) & 1) continue;
        const int o = n - 4 * f - 3 * t - 2 * w;
        const double cost = f * c.of[4] + t * c.of[3] + w * c.of[2] + o * c.of[1];
        if (take[1] >= 0 && cost >= best) continue;
        best = cost;
        take[1] = o;
        take[2] = w;
        take[3] = t;
        take[4] = f;
      }
  for (int k = 1; k <= 4; ++k) launches[k] += take[k];
}

// v of the next lane (y + 1) / of the previous one (y - 1); 0 past the ends
template <class C>
__device__ __forceinline__ C lane_up(C v) {
  if constexpr (sizeof(C) == 4) {
    return __builtin_bit_cast(
        C, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
  } else {
    typedef int I2 __attribute__((ext_vector_type(2)));
    I2 w = __builtin_bit_cast(I2, v);
    w[0] = __builtin_amdgcn_mov_dpp(w[0], 0x130, 0xf, 0xf, true);
    w[1] = __builtin_amdgcn_mov_dpp(w[1], 0x130, 0xf, 0xf, true);
    return __builtin_bit_cast(C, w);
  }
}
template <class C>
__device__ __forceinline__ C lane_down(C v) {
  if constexpr (sizeof(C) == 4) {
    return __builtin_bit_cast(
        C, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
  } else {
    typedef int I2 __attribute__((ext_vector_type(2)));
    I2 w = __builtin_bit_cast(I2, v);
    w[0] = __builtin_amdgcn_mov_dpp(w[0], 0x138, 0xf, 0xf, true);
    w[1] = __builtin_amdgcn_mov_dpp(w[1], 0x138, 0xf, 0xf, true);
    return __builtin_bit_cast(C, w);
  }
}

// What stage s keeps of its input: row X (the newest one) as far as it
// enters row X's own update.  Directions in the order of Lat<9>: e_x = -1:
// 1, 5, 6; e_x = 0: 0, 2, 3; e_x = +1: 4, 7, 8.
// (Plain members and not arrays, here and below: the compiler keeps a small
// array that meets a branch as one block of registers and copies all of it.)
template <class C>
struct SweepRow {
  C z0, z2, z3;     // pulled (or bounced) along the row
  C u4, u7, u8;     // pulled (or bounced) from row X - 1
  C o4, o7, o8;     // row X's own e_x = +1 values: what its e_x = -1 links
                    // bounce to, and what row X + 1 pulls
  uint32_t m;       // link mask of the node in row X
  uint32_t h;       // its hash (stochastic rounding)
};

// The nine values of a node.
template <class T>
struct Nine {
  T v0, v1, v2, v3, v4, v5, v6, v7, v8;
};

// One row of one lattice as it lies in memory: this lane's node.
template <int S>
struct SweepLoad {
  Nine<typename Store<S>::T> raw;
  uint32_t m, own;
};

template <int S>
__device__ __forceinline__ void sweep_load(const Grid& g,
                                           const typename Store<S>::T* __restrict__ A,
                                           const uint32_t* __restrict__ mask, uint32_t n,
                                           SweepLoad<S>& ld) {
  using T = typename Store<S>::T;
  ld.own = pidx<9>(n, 0);
  if constexpr (sizeof(T) == 8)
    ld.m = gload(mask + n);
  else
    ld.m = gload(elem((const uint16_t*)(mask + g.n), n));
  const T* a = elem(A, ld.own);
  ld.raw.v0 = gload(a);
  ld.raw.v1 = gload(a + 1 * kTile);
  ld.raw.v2 = gload(a + 2 * kTile);
  ld.raw.v3 = gload(a + 3 * kTile);
  ld.raw.v4 = gload(a + 4 * kTile);
  ld.raw.v5 = gload(a + 5 * kTile);
  ld.raw.v6 = gload(a + 6 * kTile);
  ld.raw.v7 = gload(a + 7 * kTile);
  ld.raw.v8 = gload(a + 8 * kTile);
}

// The unit `u` of a lattice: K steps of its rows, read from A, written to B.
template <int S, int K, int FORCE, class Par>
__device__ __forceinline__ void sweep_rows(const Grid& g, const SweepPlan& pl,
                                           const typename Store<S>::T* __restrict__ A,
                                           typename Store<S>::T* __restrict__ B,
                                           const uint32_t* __restrict__ mask,
                                           const Par& p, uint32_t u) {
#pragma clang fp contract(on)
  using St = Store<S>;
  using T = typename St::T;
  using C = typename St::C;
  constexpr int H = (int)kSweepHalo;
  static_assert(K <= H, "the strips keep kSweepHalo lanes");
  constexpr uint32_t kSolid = sizeof(T) == 8 ? LBM_MASK_SOLID : kMask16Solid;
  constexpr uint32_t kLid = sizeof(T) == 8 ? LBM_MASK_LID : kMask16Lid;
  const StepCoef<C>& cf = step_coef<S>(p);
  const int lane = (int)(threadIdx.x & 63u);
  const uint32_t cg = u / pl.strips;
  const int strip = (int)(u - cg * pl.strips);
  // this lane's chunk and place in the strip
  int grp = 0, pos = lane;
  if (pl.groups > 1) {
    grp = lane / (int)pl.group;
    pos = lane - grp * (int)pl.group;
  }
  const int nx = (int)g.nx, ny = (int)g.ny;
  const bool wrap_y = (g.flags & kWrapY) != 0, wrap_x = (g.flags & kWrapX) != 0;
  int y;
  bool out;
  if (wrap_y) {
    const int q = strip * (int)pl.stride + pos - H;  // -H .. ny + H + 63
    y = q % ny;
    y = y < 0 ? y + ny : y;
    out = pos >= H && pos < H + (int)pl.stride && q < ny;
  } else {
    y = strip * (int)pl.stride + pos;
    const bool last = strip + 1 == (int)pl.strips;
    out = pos >= (strip ? H : 0) && (last ? y < ny : pos < 64 - H);
    y = y < ny ? y : ny - 1;
  }
  const int rows = (int)pl.rows;
  const int xs = ((int)cg * (int)pl.groups + grp) * rows;  // first output row
  out = out && grp < (int)pl.groups && pos < (int)pl.group;
  // rows that this lane stores
  int left = out ? (xs + rows < nx ? rows : nx - xs) : 0;
  // rows xs - K .. xs + rows + K - 1 are read; beyond a walled end the end
  // row itself (its links from there bounce, so it is not used)
  int xr = xs - K;
  if (wrap_x) {
    xr %= nx;
    xr = xr < 0 ? xr + nx : xr;
  }
  auto load_row = [&](SweepLoad<S>& ld) {
    const int c = wrap_x ? xr : (xr < 0 ? 0 : (xr < nx ? xr : nx - 1));
    sweep_load<S>(g, A, mask, (uint32_t)y + __umul24((uint32_t)c, g.ny), ld);
    ++xr;
    if (wrap_x) xr = xr == nx ? 0 : xr;
  };
  uint32_t n_out = (uint32_t)y + __umul24((uint32_t)xs, g.ny);

  SweepRow<C> st[K];
#pragma unroll
  for (int s = 0; s < K; ++s) {
    st[s].z0 = st[s].z2 = st[s].z3 = st[s].u4 = st[s].u7 = st[s].u8 = (C)0;
    st[s].o4 = st[s].o7 = st[s].o8 = (C)0;
    st[s].m = st[s].h = 0u;
  }
  // bit s: the row that is new to stage s holds a node with a bounced link
  // / next to the moving wall / solid (for the whole wavefront: scalar)
  uint32_t bounced = 0, lids = 0, solids = 0;
  // t: row of the chunk that arrives.  Rows 2 s and 2 s + 1 are the first
  // that reach stage s right; from row 2 s + 2 on it forms rows.  part:
  // only the stages that do so take part (rows below 2 K).
  auto row_step = [&](int t, auto part, const SweepLoad<S>& ld, SweepLoad<S>& next) {
    constexpr bool kPart = decltype(part)::value;
    Nine<C> P{St::cvt_u(ld.raw.v0), St::cvt_u(ld.raw.v1), St::cvt_u(ld.raw.v2),
              St::cvt_u(ld.raw.v3), St::cvt_u(ld.raw.v4), St::cvt_u(ld.raw.v5),
              St::cvt_u(ld.raw.v6), St::cvt_u(ld.raw.v7), St::cvt_u(ld.raw.v8)};
    uint32_t m = ld.m;
    uint32_t h = FORCE && St::kShifted ? sr_node_hash(ld.own) : 0u;
    bounced = bounced << 1 | (__any((m & 0x1FEu) != 0u) ? 1u : 0u);
    lids = lids << 1 | (__any((m & kLid) != 0u) ? 1u : 0u);
    solids = solids << 1 | (__any((m & kSolid) != 0u) ? 1u : 0u);
    // the next row's loads run under this row's work (the last one's are
    // not used: its row is in the lattice too)
    load_row(next);
    T res[9];
#pragma unroll
    for (int s = 0; s < K; ++s) {
      SweepRow<C>& r = st[s];
      const bool form = !kPart || t >= 2 * s + 2;
      const uint32_t mx = r.m, hx = r.h;
      C g0 = r.z0, g2 = r.z2, g3 = r.z3, g4 = r.u4, g7 = r.u7, g8 = r.u8;
      C g1 = P.v1, g5 = lane_up(P.v5), g6 = lane_down(P.v6);
      if ((bounced >> (s + 1)) & 1u) {
        g1 = pick(mx, 1, r.o4, g1);
        g5 = pick(mx, 5, r.o8, g5);
        g6 = pick(mx, 6, r.o7, g6);
      }
      // the new row
      r.u4 = r.o4;
      r.u7 = lane_up(r.o7);
      r.u8 = lane_down(r.o8);
      r.z0 = P.v0;
      r.z2 = lane_up(P.v2);
      r.z3 = lane_down(P.v3);
      r.o4 = P.v4;
      r.o7 = P.v7;
      r.o8 = P.v8;
      if ((bounced >> s) & 1u) {
        r.z2 = pick(m, 2, P.v3, r.z2);
        r.z3 = pick(m, 3, P.v2, r.z3);
        r.u4 = pick(m, 4, P.v1, r.u4);
        r.u7 = pick(m, 7, P.v6, r.u7);
        r.u8 = pick(m, 8, P.v5, r.u8);
      }
      r.m = m;
      r.h = h;
      if (kPart && !form) return;
      m = mx;
      h = hx;
      // the moving-wall term, as std_collide_node adds it
      if ((lids >> (s + 1)) & 1u) {
        const uint32_t ml = (mx & kLid) ? mx : 0u;
        auto wall = [&](int i) { return pick(ml, i, cf.lid[i], (C)0); };
        g1 += wall(1);
        g2 += wall(2);
        g3 += wall(3);
        g4 += wall(4);
        g5 += wall(5);
        g6 += wall(6);
        g7 += wall(7);
        g8 += wall(8);
      }
      C gv[9] = {g0, g1, g2, g3, g4, g5, g6, g7, g8};
      // solid nodes hold the rest state only where it is stored: no fluid
      // node reads them
      std_collide_node<9, S, false, FORCE, 0>(
          p, gv, mx, false, [&](auto fd, int i, auto o) {
            if constexpr (decltype(fd)::value)
              res[i] = St::round_sr_u(o, sr_key(hx, i));
            else
              res[i] = round_out<S>(o);
          });
      if (s + 1 < K) {
        P = Nine<C>{St::cvt_u(res[0]), St::cvt_u(res[1]), St::cvt_u(res[2]),
                    St::cvt_u(res[3]), St::cvt_u(res[4]), St::cvt_u(res[5]),
                    St::cvt_u(res[6]), St::cvt_u(res[7]), St::cvt_u(res[8])};
      } else if (!kPart) {
        // row xs + t - 2 K after K steps
        if (left > 0) {
          T* b = elem(B, pidx<9>(n_out, 0));
          const bool sol = ((solids >> K) & 1u) && (mx & kSolid);
#pragma unroll
          for (int i = 0; i < 9; ++i) {
            gstore(b + i * kTile, sol ? St::rest(i, Lat<9>::W[i]) : res[i]);
          }
        }
        --left;
        n_out += g.ny;
      }
    }
  };
  // two rows per turn: the registers of the rows in flight swap roles
  // instead of being copied
  SweepLoad<S> la, lb;
  load_row(la);
  for (int t = 0; t < 2 * K; t += 2) {
    row_step(t, Forced<true>{}, la, lb);
    row_step(t + 1, Forced<true>{}, lb, la);
  }
  for (int t = 0; t < rows; t += 2) {
    row_step(t, Forced<false>{}, la, lb);
    row_step(t, Forced<false>{}, lb, la);
  }
}

template <int S, int K, class Par>
__device__ __forceinline__ void sweep_unit(const Grid& g, const SweepPlan& pl,
                                           const typename Store<S>::T* __restrict__ A,
                                           typename Store<S>::T* __restrict__ B,
                                           const uint32_t* __restrict__ mask,
                                           const Par& p, uint32_t u) {
  if (step_coef<S>(p).forced)
    sweep_rows<S, K, 1>(g, pl, A, B, mask, p, u);
  else
    sweep_rows<S, K, 0>(g, pl, A, B, mask, p, u);
}

// Calls fn(QS<9, S>{}, integral_constant<int, K>{}) for a sweep of k steps
// (2 to 4) of a D2Q9 lattice with this storage.
template <class Fn>
int dispatch_sweep(int storage, int k, Fn&& fn) {
  auto by_k = [&](auto tag) {
    if (k == 4)
      fn(tag, std::integral_constant<int, 4>{});
    else if (k == 3)
      fn(tag, std::integral_constant<int, 3>{});
    else
      fn(tag, std::integral_constant<int, 2>{});
    return LBM_OK;
  };
  if (k < 2 || k > 4) return fail(LBM_ERR_INVALID, "a sweep takes 2 to 4 steps");
  switch (storage) {
    case kStoreF32Shifted: return by_k(QS<9, kStoreF32Shifted>{});
    case LBM_STORE_F64: return by_k(QS<9, LBM_STORE_F64>{});
    case LBM_STORE_F16: return by_k(QS<9, LBM_STORE_F16>{});
    case LBM_STORE_BF16: return by_k(QS<9, LBM_STORE_BF16>{});
    default: return fail(LBM_ERR_UNSUPPORTED, "storage not built");
  }
}

}  // namespace lbm
