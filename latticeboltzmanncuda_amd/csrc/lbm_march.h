// Two steps of a large D3Q19 lattice in one pass over memory.
//
// One step at a time, FP32 and FP64 lattices are bound by the bytes they
// move, whether these come from HBM or from the Infinity Cache (128^3 and
// 256 x 128 x 128 FP32 both run at 5.8 TB/s).  Here a workgroup takes a
// column of rows x width nodes in y and z, one per thread, and marches it
// along x plane by plane: the first step of plane X reads its populations
// from memory and leaves the results in LDS, from where the neighbours'
// values of the second step are read; with those of X known, plane X - 1
// takes its second step and is written.  What a plane keeps until then stays
// in registers: the values pulled along the plane, those pulled from the
// plane before, and its own ones that its links to the plane behind bounce
// to.  Two planes' buffers in turn: one barrier a plane.  The next plane's
// loads are issued before the second step, and its link masks one plane
// earlier still, so that neither waits for the other.
//
// What it costs: the outermost rows (and, where a row does not fit, the ends
// in z) are computed by two workgroups, and so is a plane at each end of a
// chunk.  256 x 128 x 128 (8 rows of 128 nodes, 6 stored; 24 planes a chunk):
// 1.45 first steps a node.  It is bound by vector instructions then: 467 a
// step of 64 nodes, whose issue takes 50 of the 70 us; the rest is waiting at
// the planes' barriers and 94 % of the CUs at work.
//
// Per step, one at a time against this, sphere channels: FP32 256 x 128 x
// 128 108.6 -> 69.9 us, 128^3 56.3 -> 38.4, 100^3 28.5 -> 20.6, 200^3 211 ->
// 165, 80^3 15.2 -> 13.9; FP64 256 x 128 x 128 217 -> 150, 121 x 67 x 93
// 37.3 -> 28, 80^3 26.4 -> 20.5.  Not for 16 bits, whose single steps move
// half the bytes for the same instructions (256^3 FP16 212 against 238 us),
// and not for D3Q27, whose planes leave LDS for half the nodes.
//
// The per-node arithmetic is std_collide_node on the same inputs, rounded to
// the stored type between the steps: the same bytes as single steps.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "lbm_step_node.h"

namespace lbm {

// How a lattice is cut: columns of `rows` x `width` threads in y and z, with
// a rim of one node at each end in y, and in z where several strips share a
// row; marched along x in chunks of `planes`.
struct MarchPlan {
  uint32_t width, rows;
  uint32_t strips, bands;   // columns along z and y
  uint32_t planes, chunks;  // output planes of a chunk
};

// Two planes of 18 directions fill a CU's LDS: 147 KB (512 threads of FP64
// also need twice the registers).
inline constexpr int march_threads(size_t bytes) { return bytes == 8 ? 512 : 1024; }
constexpr uint32_t kMarchSlots = 256;  // one workgroup a CU

// The cheapest cut of a lattice, and its cost: threads' plane steps per node
// (a node on its own would cost 1).  A plane's rim rows and ends count, the
// three planes by which a chunk's march is longer than its output, and the
// last round of workgroups, which may be nearly empty.  Strips have
// short rows that start anywhere in a cache line: a thread's step is 1.4
// times as dear (200^3 FP32, 1 strip 165 us at a cost of 2.1, 2 strips 155 at
// 1.4; 256 x 128 x 128 FP64 150 at 2.1, 4 strips 151 at 1.44), for FP64 with
// rows that are no whole tiles either 1.15 times (121 x 67 x 93, 31 us at 2.4
// and 4 strips 28 at 1.9).
inline MarchPlan march_plan(const Grid& g, size_t bytes, double* cost) {
  const uint32_t threads = (uint32_t)march_threads(bytes);
  MarchPlan best{};
  *cost = 1e300;
  for (uint32_t strips = 1; strips <= 64; ++strips) {
    MarchPlan p{};
    p.strips = strips;
    p.width = strips == 1 ? g.nz : (g.nz + strips - 1) / strips + 2;
    if (strips > 1 && p.width < 24) break;
    p.rows = threads / p.width;
    p.rows = p.rows < g.ny + 2 ? p.rows : g.ny + 2;
    if (p.rows < 3) continue;
    p.bands = (g.ny + p.rows - 3) / (p.rows - 2);
    const uint64_t columns = (uint64_t)p.strips * p.bands;
    const double dear = strips == 1 ? 1.0 : bytes == 4 || g.nz % kTile == 0 ? 1.4 : 1.15;
    // as many chunks as fill whole rounds of workgroups
    for (uint64_t rounds = 1; rounds <= 64; ++rounds) {
      uint64_t chunks = rounds * kMarchSlots / columns;
      if (chunks == 0) continue;
      chunks = chunks < g.nx ? chunks : g.nx;
      p.planes = (uint32_t)((g.nx + chunks - 1) / chunks);
      p.chunks = (g.nx + p.planes - 1) / p.planes;
      const uint64_t taken = (columns * p.chunks + kMarchSlots - 1) / kMarchSlots;
      const double c = (double)(taken * kMarchSlots * threads) * (p.planes + 3) * dear / g.n;
      if (c < *cost) {
        *cost = c;
        best = p;
      }
      if (p.planes < 8) break;
    }
  }
  return best;
}

// Where the march is taken: 64^3 FP32 8.3 us one step at a time, 10.3 so
// (cost 5), FP64 13.6 and 13.9 (3.0); 64 x 100 x 60 FP64 20.1 and 17.5.  A
// cost of 1 is about 9.5 ps a node FP32 and 17 FP64, a single step 26-30 and
// 50-54, the more the smaller the lattice.
constexpr uint32_t kMarchMinNodes = 350000, kMarchLargeNodes = 2000000;
inline bool march_pays(const Grid& g, size_t bytes, double cost) {
  if (population_elems(19, g.n) * bytes >> 32) return false;  // 32-bit byte offsets
  return cost <= (g.n < kMarchLargeNodes ? 3.1 : 2.6);
}

template <class T>
struct MarchShared {
  // directions 1..18 of a plane, two planes in turn
  T val[2][18][march_threads(sizeof(T))];
};

// A plane's populations as they are pulled (or bounced) for its first step.
template <class T>
struct MarchLoad {
  T raw[19];
  uint32_t m, own;  // the node's mask word and element index
};

// Chunk u of a lattice's columns (chunks of the same planes first, along z,
// then y): two steps, read from A, written to B.  NT: non-temporal stores.
template <int S, bool LID, bool NT>
__device__ __forceinline__ void march_unit(const Grid& g, const MarchPlan& pl,
                                           const typename Store<S>::T* __restrict__ A,
                                           typename Store<S>::T* __restrict__ B,
                                           const uint32_t* __restrict__ mask,
                                           const StepCoef<typename Store<S>::C>& p,
                                           MarchShared<typename Store<S>::T>& sh, uint32_t u) {
  constexpr int Q = 19;
  using L = Lat<Q>;
  using St = Store<S>;
  using T = typename St::T;
  using C = typename St::C;
  const uint32_t per_chunk = pl.strips * pl.bands;
  const uint32_t chunk = u / per_chunk;
  const uint32_t rest = u - chunk * per_chunk;
  const uint32_t band = rest / pl.strips, strip = rest - band * pl.strips;
  const int t = (int)threadIdx.x;
  const int w = (int)pl.width;
  int ty = t / w;
  const int tz = t - ty * w;
  const bool live = ty < (int)pl.rows;  // spare threads repeat the last row
  const int tt = live ? t : t - w * (ty - (int)pl.rows + 1);
  ty = live ? ty : (int)pl.rows - 1;
  const int nx = (int)g.nx, ny = (int)g.ny, nz = (int)g.nz;
  const bool one = pl.strips == 1;
  int z = one ? tz : (int)strip * (w - 2) + tz - 1;
  int y = (int)band * ((int)pl.rows - 2) + ty - 1;
  const bool out = live && ty > 0 && ty + 1 < (int)pl.rows && y < ny &&
                   (one || (tz > 0 && tz + 1 < w && z < nz));
  // rim coordinates wrapped or, beyond a wall (not used there), held inside
  auto fold = [](int v, int n, bool wrap) {
    if (wrap) {
      v %= n;
      return v < 0 ? v + n : v;
    }
    return v < 0 ? 0 : (v < n ? v : n - 1);
  };
  y = fold(y, ny, g.flags & kWrapY);
  z = fold(z, nz, g.flags & kWrapZ);
  const uint32_t plane = g.ny * g.nz;
  // the column's source columns in bytes, wrapped along each axis
  const uint32_t row = g.nz * (uint32_t)sizeof(T);
  const uint32_t cy[3] = {(uint32_t)(y + 1 == ny ? 0 : y + 1) * row, (uint32_t)y * row,
                          (uint32_t)(y == 0 ? ny - 1 : y - 1) * row};
  const uint32_t cz[3] = {(uint32_t)(z + 1 == nz ? 0 : z + 1) * (uint32_t)sizeof(T),
                          (uint32_t)z * (uint32_t)sizeof(T),
                          (uint32_t)(z == 0 ? nz - 1 : z - 1) * (uint32_t)sizeof(T)};
  // LDS places of the neighbours: wrapped where a strip is a whole row, else
  // held inside (a rim's second step is not used)
  auto place = [&](int a, int b) {  // source of e_y = a, e_z = b
    int sy = ty - a, sz = tz - b;
    sy = sy < 0 ? 0 : (sy < (int)pl.rows ? sy : (int)pl.rows - 1);
    if (one)
      sz = sz < 0 ? w - 1 : (sz < w ? sz : 0);
    else
      sz = sz < 0 ? 0 : (sz < w ? sz : w - 1);
    return sy * w + sz;
  };
  const int pzm = place(0, 1), pzp = place(0, -1), pym = place(1, 0), pyp = place(-1, 0);
  auto nb = [&](int i) {
    const int a = L::E[i][1], b = L::E[i][2];
    if (a == 0) return b == 0 ? tt : (b > 0 ? pzm : pzp);
    if (b == 0) return a > 0 ? pym : pyp;
    return (a > 0 ? pym : pyp) + (b > 0 ? pzm : pzp) - tt;
  };
  const bool wrap_x = (g.flags & kWrapX) != 0;
  const int xs = (int)(chunk * pl.planes);
  const int xe = xs + (int)pl.planes < nx ? xs + (int)pl.planes : nx;
  auto fold_x = [&](int X) { return (uint32_t)fold(X, nx, wrap_x); };
  auto mask_of = [&](int X) {
    return gload(mask + (fold_x(X) * plane + (cy[1] + cz[1]) / (uint32_t)sizeof(T)));
  };
  // Populations in byte offsets (below 2^32: march_pays) through a buffer
  // resource: element (n, i) lies at v + v / kRow (Q - 1) kRow + i kRow, v
  // being n in bytes, so a pulled address takes an add, a shift and one 24-bit
  // multiply-add, and a bounced one two more (its part of i kRow that both
  // share is the load's constant): 114 instructions a node instead of the 193
  // of 64-bit addresses from element indices.
  constexpr uint32_t kRow = kTile * (uint32_t)sizeof(T);
  const auto from = buffer_rsrc(A, (g.n + kTile - 1) / kTile * (Q * kRow));
  auto load = [&](uint32_t at, uint32_t shift) -> T {
    const int off = (int)(at + shift % 4096u), rest = (int)(shift / 4096u * 4096u);
    if constexpr (sizeof(T) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(from, off, rest, 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(from, off, rest, 0));
  };
  auto gather = [&](int X, uint32_t m, MarchLoad<T>& ld) {
    constexpr uint32_t kSize = (uint32_t)sizeof(T);
    const uint32_t x0 = fold_x(X);
    const uint32_t bx[3] = {(x0 + 1 == g.nx ? 0u : x0 + 1) * plane * kSize, x0 * plane * kSize,
                            (x0 == 0 ? g.nx - 1 : x0 - 1) * plane * kSize};
    auto pull = [&](int i) {
      const uint32_t v = bx[L::E[i][0] + 1] + cy[L::E[i][1] + 1] + cz[L::E[i][2] + 1];
      return __umul24(v / kRow, (Q - 1) * kRow) + v;
    };
    ld.m = m;
    const uint32_t own = pull(0);
    ld.own = own / kSize;
    if (__any((m & ((1u << Q) - 2u)) != 0u)) {
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const uint32_t lo = (uint32_t)(i < L::INV[i] ? i : L::INV[i]) * kRow;
        const uint32_t a = pull(i) + ((uint32_t)i * kRow - lo);
        const uint32_t b = own + ((uint32_t)L::INV[i] * kRow - lo);
        ld.raw[i] = load(i ? select_bit(m, i, b, a) : a, lo);
      }
    } else {
#pragma unroll
      for (int i = 0; i < Q; ++i) ld.raw[i] = load(pull(i), (uint32_t)i * kRow);
    }
  };
  const bool any_out = __any(out);
  // plane X - 1 as far as it is known: pulled along it and from X - 2; un:
  // what plane X pulls from X - 1; o: plane X - 1's own e_x = +1 values
  C r[Q], un[Q], o[Q];
  uint32_t mr = 0, ownr = 0;
#pragma unroll
  for (int i = 0; i < Q; ++i) r[i] = un[i] = o[i] = (C)0;
  uint32_t mnext = mask_of(xs);
  MarchLoad<T> ld;
  gather(xs - 1, mask_of(xs - 1), ld);
  // (two planes a turn, without copies of the loads in flight, spill
  // registers: 256 x 128 x 128 FP32 105 us)
  for (int X = xs - 1; X <= xe; ++X) {
    // plane X's first step (what solid nodes get is not read: the links to them
    // bounce)
    C gv[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) gv[i] = St::cvt_u(ld.raw[i]);
    const uint32_t m = ld.m & ~LBM_MASK_SOLID, own = ld.own;
    const bool solid = (ld.m & LBM_MASK_SOLID) != 0u;
    T f1[Q];
    std_collide_node<Q, S, LID, 2, 0>(p, gv, m, false, [&](auto fd, int i, auto v) {
      if constexpr (decltype(fd)::value)
        f1[i] = St::round_sr_u(v, sr_key(St::kShifted ? sr_node_hash(own) : 0u, i));
      else
        f1[i] = round_out<S>(v);
    });
    auto& buf = sh.val[X & 1];
    if (live) {
#pragma unroll
      for (int i = 1; i < Q; ++i) buf[i - 1][t] = f1[i];
    }
    // the next plane's loads run under the second step
    if (X < xe) {
      const uint32_t m1 = mnext;
      mnext = mask_of(X + 2);
      gather(X + 1, m1, ld);
    }
    __syncthreads();
    if (any_out) {
      // plane X - 1: what comes from plane X
      if (X > xs) {
        C h[Q];
#pragma unroll
        for (int i = 0; i < Q; ++i) {
          if (L::E[i][0] < 0) {
            const C v = St::cvt_u(buf[i - 1][nb(i)]);
            h[i] = pick(mr, i, o[L::INV[i]], v);
          } else {
            h[i] = r[i];
          }
        }
        const uint32_t m2 = mr & ~LBM_MASK_SOLID;
        T* const b = elem(B, ownr);
        std_collide_node<Q, S, LID>(p, h, m2, (mr & LBM_MASK_SOLID) != 0u,
                                    [&](auto fd, int i, auto v) {
          T res;
          if constexpr (decltype(fd)::value)
            res = St::round_sr_u(v, sr_key(St::kShifted ? sr_node_hash(ownr) : 0u, i));
          else
            res = round_out<S>(v);
          if (out) {
            if (NT)
              gstore_nt(b + i * kTile, res);
            else
              gstore(b + i * kTile, res);
          }
        });
      }
      // plane X
      const uint32_t mx = solid ? m | LBM_MASK_SOLID : m;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        if (i == 0) {
          r[i] = St::cvt_u(f1[0]);
        } else if (L::E[i][0] == 0) {
          const C v = St::cvt_u(buf[i - 1][nb(i)]);
          r[i] = pick(mx, i, St::cvt_u(f1[L::INV[i]]), v);
        } else if (L::E[i][0] > 0) {
          r[i] = pick(mx, i, St::cvt_u(f1[L::INV[i]]), un[i]);
          un[i] = St::cvt_u(buf[i - 1][nb(i)]);
          o[i] = St::cvt_u(f1[i]);
        }
      }
      mr = mx;
      ownr = own;
    }
  }
}

}  // namespace lbm
