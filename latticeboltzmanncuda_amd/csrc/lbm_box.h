// Several steps of a small D2Q9 lattice in one launch, box by box in LDS.
//
// A small lattice stepped one launch at a time pays for the launch, a chain
// of dependent loads (constants, link mask, populations) and the store that
// the next launch waits for, and hardly for its arithmetic.  Here a
// workgroup takes a box of kSide x kSide nodes: its first step reads the
// nodes within K - 1 of the box from memory (std_gather) and leaves them in
// LDS, the following ones work on a region one node narrower each, from LDS
// to LDS, and the last writes the box.  Neighbouring boxes compute their
// common rims twice, so nothing is exchanged between workgroups.  The
// populations of two steps lie in two buffers: one barrier a step.
//
// Per step on MI355X, one launch a step (from 512^2 on: four steps in one
// sweep) against this, FP32 cavity: 128^2 3.5-4.2 -> 1.06 us, 256^2 3.6 ->
// 1.39, 512^2 4.6 -> 2.96, 800^2 6.3 -> 5.9; FP64 256^2 4.8 -> 1.87, FP16
// channel 256^2 4.4 -> 1.7.  What is left at 128^2 is latency: per launch
// about 2.5 us of start, loads and store, and 0.7 us a step of one chain of
// LDS reads and collision.
//
// (Batches keep their tiles: with boxes, which fit their lattices badly, a
// step of eight FP16 lattices of 64 to 512 a side took 5.15 us instead of
// 5.43, of 64 lattices of 32 to 300 a side 10.0 instead of 9.3.)
//
// The per-node arithmetic is std_collide_node on the same inputs, rounded to
// the stored type between steps, so K steps give the same bytes as K single
// ones.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "lbm_step_node.h"
#include "lbm_sweep.h"

namespace lbm {

// kSide x kSide output nodes, K steps; kWidth: side of the first step's
// region.
template <int K_, int SIDE>
struct Box {
  static constexpr int K = K_, kSide = SIDE, kRim = K - 1, kWidth = SIDE + 2 * kRim;
  static constexpr int kCells = kWidth * kWidth;
  static constexpr int kThreads = (kCells + 63) / 64 * 64;
  static_assert(kThreads <= 1024, "a region takes one thread per cell");
};

// K = 8 saves launches and loads, K = 4 computes less of the rims twice
// (256^2 FP32 1.39 against 1.93 us per step, 512^2 3.26 against 2.96); a
// side of 8 gives a small lattice more workgroups (128^2: 256 of them, 1.06
// against 1.21 us).
using BoxTiny = Box<8, 8>;
using BoxSmall = Box<8, 16>;
template <int K>
using BoxWide = Box<K, 16>;  // K = 2 to 4
constexpr uint32_t kBoxTinyNodes = 24000;
// FP64 computes its rims at half the rate (330^2: 3.34 us per step with 8
// steps, 3.20 with 4; FP32 1.89 and 2.83)
inline uint32_t box_small_nodes(int storage) {
  return storage_bytes(storage) == 8 ? 80000u : 130000u;
}
// Up to here boxes are faster than sweeps (FP32 800^2 5.9 against 6.3 us,
// 1000^2 8.3 / 7.5; FP64 620^2 6.4 / 7.4, 800^2 10.0 / 8.5) or, with 16 bits,
// than single steps (800^2 5.2-6.6 against 5.8-7.0, 1000^2 7.4-9.5 /
// 7.5-9.4).
inline uint32_t box_max_nodes(int storage) {
  return storage_bytes(storage) == 8 ? 500000u : storage_bytes(storage) == 4 ? 700000u : 800000u;
}
// Workgroups of BoxWide for a lattice; the limits above count the nodes of
// its whole boxes (a lattice one node wide would fill a sixteenth of them).
inline uint64_t box_wide_count(const Grid& g) {
  return (uint64_t)((g.nx + 15) / 16) * ((g.ny + 15) / 16);
}
constexpr uint32_t kBoxWideNodes = 16 * 16;

// Microseconds of a launch of k steps, k of 1 (one step of the lattice by
// itself) to 4 (BoxWide), fitted to what lattices of 64^2 to 800^2 and thin
// ones of 20000 x 8 to 60 x 6000 took: a launch of boxes is its start and
// load latency and so much a box, little less where part of it lies outside
// the lattice.  So short calls and thin lattices go by single steps where
// these are faster (FP16 520 x 990 by twos 7.7-8.3 us a step, by threes
// 5.9-6.9, by fours 4.8-5.7, singly 4.8-6.0; FP32 20000 x 20 by twos 7.2, by
// fours 5.1, singly 5.9).
inline StepCosts box_costs(int storage, const Grid& g) {
  const double n = g.n, whole = (double)(box_wide_count(g) * kBoxWideNodes);
  const double boxes = (0.6 * whole + 0.4 * n) / kBoxWideNodes;
  auto most = [](double a, double b) { return a > b ? a : b; };
  switch (storage_bytes(storage)) {
    case 2:
      // (two and three with a margin: where single steps are bound by the host,
      // they take 2.7 to 3.6 us, as the host's clock is)
      return {{0.0, most(3.15, 1.2 + 8.5e-6 * n), 1.2 * (5.5 + 0.0050 * boxes),
               1.1 * (5.4 + 0.0064 * boxes), 5.8 + 0.0066 * boxes}};
    case 8:
      return {{0.0, most(3.7, 2.0 + 24e-6 * n), 5.2 + 0.0098 * boxes, 6.5 + 0.0115 * boxes,
               7.5 + 0.0127 * boxes}};
    default:
      return {{0.0, most(3.3, 2.6 + 10e-6 * n), 4.6 + 0.0056 * boxes, 5.8 + 0.0067 * boxes,
               6.5 + 0.0072 * boxes}};
  }
}

// Thin lattices fill little of their boxes, whose cells beyond a wall idle:
// where that leaves more than two boxes a CU, single steps are faster below a
// fifth (per step singly / by boxes, FP32 40000 x 1 3.2 / 7.4 us, 2 x 50000
// 3.4 / 3.9, 5000 x 4 3.3 / 1.3) and fours than eights below six tenths (FP64
// 10000 x 8 singly 4.5, by eights 4.9).
constexpr uint64_t kBoxesAny = 512;
inline bool box_fits(const Grid& g) {
  const uint64_t boxes = box_wide_count(g);
  return boxes <= kBoxesAny || boxes * kBoxWideNodes <= 5ull * g.n;
}
inline bool box_eights_fit(const Grid& g) {
  const uint64_t boxes = box_wide_count(g);
  return boxes <= kBoxesAny || 6 * boxes * kBoxWideNodes <= 10ull * g.n;
}

template <class X, class T>
struct BoxShared {
  T val[2][9][X::kCells];
  uint32_t link[X::kCells];  // a cell's link mask, kBoxSolid, kBoxOutside
  uint32_t axis[2 * X::kWidth];
};
// axis[]: the rows' x times ny and the columns' y, wrapped, or this where
// they lie beyond a wall; link[] of such a cell
constexpr uint32_t kBoxOutside = 1u << 29;
constexpr uint32_t kBoxSolid = 1u << 28;

// Step s (1..K) of the box whose first row and column are x0 and y0.
template <class X, int S, int s, class P>
__device__ __forceinline__ void box_steps(const Grid& g, const typename Store<S>::T* __restrict__ A,
                                          typename Store<S>::T* __restrict__ B,
                                          const uint32_t* __restrict__ mask,
                                          const uint32_t* __restrict__ cls, const P& p,
                                          BoxShared<X, typename Store<S>::T>& sh, uint32_t x0,
                                          uint32_t y0) {
  using L = Lat<9>;
  using St = Store<S>;
  using T = typename St::T;
  using C = typename St::C;
  constexpr int W = X::kWidth, d = s - 1, R = W - 2 * d;
  const int c = (int)threadIdx.x;
  if (c < R * R) {
    const int cx = c / R, cy = c - cx * R;  // in this step's region
    const int cell = (cx + d) * W + cy + d;
    const uint32_t ax = sh.axis[cx + d], ay = sh.axis[W + cy + d];
    if (!((ax | ay) & kBoxOutside)) {
      const uint32_t n = ax + ay, own = pidx<9>(n, 0);
      T raw[9];
      uint32_t m;
      bool solid;
      if constexpr (s == 1) {
        NodeLoad<9, S> ld;
        std_gather<9, S>(g, A, mask, cls, n, ld);
        m = ld.m;
        solid = ld.solid;
        sh.link[cell] = m | (solid ? kBoxSolid : 0u);
#pragma unroll
        for (int i = 0; i < 9; ++i) raw[i] = ld.raw[i];
      } else {
        // cells beyond a wall hold nothing: the links to them bounce
        const auto& from = sh.val[s & 1];
        m = sh.link[cell];
        solid = (m & kBoxSolid) != 0u;
        m &= ~kBoxSolid;
#pragma unroll
        for (int i = 0; i < 9; ++i) raw[i] = from[i][cell - (L::E[i][0] * W + L::E[i][1])];
        if (__any(m != 0u)) {
#pragma unroll
          for (int i = 1; i < 9; ++i) {
            const T back = from[L::INV[i]][cell];
            raw[i] = ((m >> i) & 1u) ? back : raw[i];
          }
        }
      }
      C gv[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) gv[i] = St::cvt_u(raw[i]);
      T res[9];
      std_collide_node<9, S, true>(p, gv, m, solid, [&](auto forced, int i, auto o) {
        if constexpr (decltype(forced)::value)
          res[i] = St::round_sr_u(o, sr_key(St::kShifted ? sr_node_hash(own) : 0u, i));
        else
          res[i] = round_out<S>(o);
        if constexpr (s < X::K) sh.val[(s + 1) & 1][i][cell] = res[i];
      });
      // a box beyond a periodic end holds nodes that another one stores
      if (s == X::K && x0 + (uint32_t)cx < g.nx && y0 + (uint32_t)cy < g.ny) {
        T* b = elem(B, own);
#pragma unroll
        for (int i = 0; i < 9; ++i) gstore(b + i * kTile, res[i]);
      }
    }
  }
  if constexpr (s < X::K) {
    __syncthreads();
    box_steps<X, S, s + 1>(g, A, B, mask, cls, p, sh, x0, y0);
  }
}

// K steps of box u of a lattice (boxes lie along y first), read from A,
// written to B.
template <class X, int S, class P>
__device__ __forceinline__ void box_unit(const Grid& g, const typename Store<S>::T* __restrict__ A,
                                         typename Store<S>::T* __restrict__ B,
                                         const uint32_t* __restrict__ mask,
                                         const uint32_t* __restrict__ cls, const P& p,
                                         BoxShared<X, typename Store<S>::T>& sh, uint32_t u) {
  const uint32_t across = (g.ny + X::kSide - 1) / X::kSide;
  const uint32_t bx = u / across;
  const uint32_t x0 = bx * X::kSide, y0 = (u - bx * across) * X::kSide;
  const int t = (int)threadIdx.x;
  if (t < 2 * X::kWidth) {
    const bool row = t < X::kWidth;
    const int len = (int)(row ? g.nx : g.ny);
    int v = (row ? (int)x0 + t : (int)y0 + t - X::kWidth) - X::kRim;
    if (g.flags & (row ? kWrapX : kWrapY)) {
      v %= len;
      v = v < 0 ? v + len : v;
    }
    sh.axis[t] = v >= 0 && v < len ? (uint32_t)v * (row ? g.ny : 1u) : kBoxOutside;
  }
  __syncthreads();
  box_steps<X, S, 1>(g, A, B, mask, cls, p, sh, x0, y0);
}

// Calls fn(box type, integral_constant<int, S>{}) for a lattice of so many
// nodes and k steps (8, or 2 to 4).
template <class Fn>
int dispatch_box(int storage, uint32_t nodes, int k, Fn&& fn) {
  auto by_k = [&](auto st) {
    if (k == 8 && nodes <= kBoxTinyNodes)
      fn(BoxTiny{}, st);
    else if (k == 8)
      fn(BoxSmall{}, st);
    else if (k == 4)
      fn(BoxWide<4>{}, st);
    else if (k == 3)
      fn(BoxWide<3>{}, st);
    else
      fn(BoxWide<2>{}, st);
    return LBM_OK;
  };
  if (k != 8 && (k < 2 || k > 4)) return fail(LBM_ERR_INVALID, "boxes take 8 or 2 to 4 steps");
  switch (storage) {
    case kStoreF32Shifted: return by_k(std::integral_constant<int, kStoreF32Shifted>{});
    case LBM_STORE_F64: return by_k(std::integral_constant<int, LBM_STORE_F64>{});
    case LBM_STORE_F16: return by_k(std::integral_constant<int, LBM_STORE_F16>{});
    case LBM_STORE_BF16: return by_k(std::integral_constant<int, LBM_STORE_BF16>{});
    default: return fail(LBM_ERR_UNSUPPORTED, "storage not built");
  }
}

}  // namespace lbm
