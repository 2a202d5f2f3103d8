// First- and second-order chains on unrefined 1-gradient lattices: the
// lattice in wave tiles, several contour steps between two barriers.
// Device code, included by scf_fused.hip after its LDS helpers.
#pragma once
#include <type_traits>

namespace nscf {

// A wave holds 64 S consecutive positions of the lattice in registers (S per
// lane); the inner 64 S - 2 H of them are its own, H on each side are a halo of its neighbours' positions.  A contour step takes the
// adjacent values from the adjacent lanes (DPP, no LDS), so the halo goes
// stale by one position per step and side, and only every H-th step the
// waves exchange their own values through LDS behind one barrier.
//
// What bounds a chain is its serial length: N steps forward and N backward,
// each waiting for the one before.  One site per thread with the row in LDS
// paid an LDS write, a barrier and an LDS read per step (second order, 400
// layers, N = 2000: 1.5 us per step).  A tile step is a few lane moves and
// the arithmetic.
//
// Positions run over 0 .. M-1, the lattice with its ghosts, and H past
// either end; a position outside the lattice stands for the site that
// set_bounds copies there, followed further by unfolding the boundary
// (tile_unfold), and evolves as that site does.
// (sizes: tile_per_lane and the like in scf_device.h)

__device__ __forceinline__ double lane_below(double v) {  // lane i reads lane i - 1
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x138, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x138, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ double lane_above(double v) {  // lane i reads lane i + 1
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x130, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// The site x that position p stands for, whether it lies there reversed
// (its lower neighbour on the upper side), and whether there is one at all
// (a surface has nothing behind it).  A mirror reverses, a periodic boundary
// does not.
template <typename Sys>
__device__ __forceinline__ void tile_unfold(const Sys &S, int p, int halo, int &x, bool &rev, bool &live) {
  const int MX = S.MX;
  const int xmin = S.surface_lo ? 0 : 1, xmax = S.surface_hi ? MX + 1 : MX;
  x = p;
  rev = false;
  live = true;
  if (p >= xmin && p <= xmax) return;
  const bool down = p < xmin;
  int n = down ? xmin - p : p - xmax;
  if (n > halo + 1) live = false;  // nothing owned depends on it
  x = down ? xmin : xmax;
  for (; live && n > 0; n--) {
    x += down != rev ? -1 : 1;
    const bool below = x < xmin, above = x > xmax;
    if (below || above) {
      const int to = below ? S.bx1 : S.bxm;
      const bool surf = below ? S.surface_lo : S.surface_hi;
      const bool mirror = below ? to == 1 : to == MX;
      if (surf) live = false;
      if (mirror) rev = !rev;
      x = to;
    }
  }
  if (!live) x = 0;
}

// kC = 1: first order (LG1Planar::propagate src/LG1Planar.cpp:146-149,
// LGrad1::propagate src/LGrad1.cpp:441-445).  kC = 3: second order, simple
// cubic, components +x, lateral, -x (LG1Planar::propagateF/B
// src/LG1Planar.cpp:57-136, LGrad1::propagateF/B src/LGrad1.cpp:285-429),
// composition weights 1/6, 4/6, 1/6, GN = (G0 + 4 G1 + G2) / 6
// (src/LGrad1.cpp:876-910, 943-955); the surface ghosts' weights are zero
// (checked by the caller).
//
// A block's rows fall into segments of kK.  The forward pass keeps the first
// row of each in memory; the backward pass recomputes a segment's rows into
// registers (f) just before it composes them, with the next segment's row
// already on its way: the rows of a 400-layer, N = 2000 second-order chain
// are 19 MB, which one compute unit cannot stream at the rate of these steps.
// The recomputation repeats the forward pass's steps.
//
// A ghost's density (only phitot on the ghosts sees it) composes Gf as
// set_bounds left it, i.e. the value of the position's site, with Gb as the
// step leaves it there before bounding: the step of the position's own value
// without what comes from beyond the lattice (on curved lattices without any
// neighbour, whose weights are zero there), with the ghost's segment weight.
// Only the waves that hold a ghost form that (kGhost); the last row counts
// zero (ComputeGN's remove_bounds, src/LGrad1.cpp:213-221,863-874).
//
// Measured on one MI355X, one system, time per row of the chain (forward and
// backward; before: one site per thread, a barrier per step): first order 100
// layers 331 -> 152 ns, 400 layers 507 -> 170 ns; second order 1657 -> 246 ns
// and 2826 -> 332 ns.  512 mixed systems (50-400 layers, N 20-2000): 0.84 ->
// 0.13 ms per evaluation on average, the slowest 6.1 -> 0.73 ms.  Two
// positions per lane for second order were tried and spill (280 B per lane
// under the 128 registers of a 1024-thread kernel), which waits for memory in
// every segment: 450 ns per step.
template <int kC, bool kCurved>
__device__ __noinline__ void chain1d_tile(const DevSys &S0, int mo) {
  constexpr int S_ = tile_per_lane(kC), H = tile_halo(kC), U = tile_own(kC), kK = tile_rows_every(kC);
  static_assert(kK <= H, "a segment fits between two exchanges");
  CSys &S = uniform_sys(S0);
  mo = __builtin_amdgcn_readfirstlane(mo);  // an argument arrives in a vector register
  const int M = S.M, MX = S.MX;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int nw = tile_waves(M, kC);
  const bool work = wave < nw;
  const int b0 = S.mol_block_begin[mo], b1 = S.mol_block_begin[mo + 1];
  const int N = S.mol_N[mo];
  const gdbl *G1 = hbm(S.G1);

  // ---- this lane's positions
  const int p0 = wave * U - H + lane * S_;
  int x[S_];
  bool rev[S_], live[S_], real[S_], halo[S_], ghost[S_];
#pragma unroll
  for (int j = 0; j < S_; j++) {
    const int p = p0 + j, at = lane * S_ + j;
    tile_unfold(S, p, H, x[j], rev[j], live[j]);
    const bool own = work && at >= H && at < H + U && p < M;
    if (!work) live[j] = false;
    real[j] = own && live[j] && x[j] == p && !rev[j];
    halo[j] = live[j] && !real[j];
    ghost[j] = own && live[j] && (p < 1 || p > MX);
  }
  bool any = false;
#pragma unroll
  for (int j = 0; j < S_; j++) any = any || ghost[j];
  const bool ghosts = __any(any);

  // ---- weights: the segment's (g1) and on curved lattices the step's to
  // smaller and larger positions (first order: lambda-, lambda0, lambda+;
  // second order: the reflection weights)
  double g1[S_], wl[S_], w0[S_], wr[S_], wl0[S_], wr0[S_];
  const double lam = S.lambda, lam0 = 1.0 - 2.0 * S.lambda;
  const double P0 = S.mol_P[mo][0], P1 = S.mol_P[mo][1], P1x4 = 4 * P1, Pm = 2 * P1 + P0;
  if constexpr (kCurved) {
#pragma unroll
    for (int j = 0; j < S_; j++) {
      const bool lo = x[j] < 1, hi = x[j] > M - 2;
      const gdbl *dn = hbm(kC == 1 ? S.lam_m : S.l_1), *up = hbm(kC == 1 ? S.lam_p : S.l1);
      const double a = lo ? 0.0 : dn[x[j]], b = hi ? 0.0 : up[x[j]];
      wl[j] = rev[j] ? b : a;
      wr[j] = rev[j] ? a : b;
      if constexpr (kC == 1) {
        w0[j] = hbm(S.lam_0)[x[j]];
      } else {
        const double a0 = lo ? 0.0 : hbm(S.l_11)[x[j]], b0 = hi ? 0.0 : hbm(S.l11)[x[j]];
        wl0[j] = rev[j] ? b0 : a0;
        wr0[j] = rev[j] ? a0 : b0;
      }
    }
  }
  auto weight = [&](int b, int j) {
    const gdbl *g = G1 + (size_t)S.block_seg[b] * M;
    return live[j] ? g[(unsigned)x[j]] : 0.0;
  };
  auto load_block = [&](int b) {
#pragma unroll
    for (int j = 0; j < S_; j++) g1[j] = weight(b, j);
  };

  // ---- one step in place; in the backward direction also the composition
  // with row f.  hl, hr: 0 where a ghost's lower / upper neighbour is left
  // out of its density, else 1.
  double racc[S_];
  double hl[S_], hr[S_];
#pragma unroll
  for (int j = 0; j < S_; j++) {
    hl[j] = ghost[j] && (kCurved || p0 + j < 1) ? 0.0 : 1.0;
    hr[j] = ghost[j] && (kCurved || p0 + j > MX) ? 0.0 : 1.0;
  }
  auto step_fwd = [&](double (&v)[kC][S_]) {
    if constexpr (kC == 1) {
      double l = lane_below(v[0][S_ - 1]);
      const double r = lane_above(v[0][0]);
#pragma unroll
      for (int j = 0; j < S_; j++) {
        const double u = j + 1 < S_ ? v[0][j + 1 < S_ ? j + 1 : j] : r;
        double t;
        if constexpr (kCurved)
          t = w0[j] * v[0][j] + wl[j] * l + wr[j] * u;
        else
          t = lam * l + lam0 * v[0][j] + lam * u;
        l = v[0][j];
        v[0][j] = t * g1[j];
      }
    } else {
      // A goes to the upper neighbour, C to the lower one
      double A[S_], C[S_];
#pragma unroll
      for (int j = 0; j < S_; j++) {
        A[j] = P0 * v[0][j] + P1x4 * v[1][j];
        C[j] = P1x4 * v[1][j] + P0 * v[2][j];
      }
      const double l = lane_below(A[S_ - 1]), r = lane_above(C[0]);
#pragma unroll
      for (int j = 0; j < S_; j++) {
        const double al = j > 0 ? A[j > 0 ? j - 1 : 0] : l;
        const double cu = j + 1 < S_ ? C[j + 1 < S_ ? j + 1 : j] : r;
        const double b = P1 * v[0][j] + Pm * v[1][j] + P1 * v[2][j];
        double a = al, c = cu;
        if constexpr (kCurved) {
          a = wl[j] * al + wl0[j] * C[j];
          c = wr[j] * cu + wr0[j] * A[j];
        }
        v[0][j] = a * g1[j];
        v[1][j] = b * g1[j];
        v[2][j] = c * g1[j];
      }
    }
  };
  constexpr double wc[3] = {1.0 / 6.0, 4.0 / 6.0, 1.0 / 6.0};
  auto step_bwd = [&](auto tag, double (&v)[kC][S_], const double (&f)[kC][S_]) {
    constexpr bool kGhost = decltype(tag)::value;
    if constexpr (kC == 1) {
      double l = lane_below(v[0][S_ - 1]);
      const double r = lane_above(v[0][0]);
#pragma unroll
      for (int j = 0; j < S_; j++) {
        const double u = j + 1 < S_ ? v[0][j + 1 < S_ ? j + 1 : j] : r;
        double t, d;
        if constexpr (kCurved)
          t = w0[j] * v[0][j] + wl[j] * l + wr[j] * u;
        else
          t = lam * l + lam0 * v[0][j] + lam * u;
        if constexpr (kGhost && !kCurved)
          d = (lam * (hl[j] * l) + lam0 * v[0][j] + lam * (hr[j] * u)) * g1[j];
        l = v[0][j];
        v[0][j] = t * g1[j];
        if constexpr (!kGhost || kCurved) d = v[0][j];  // (a curved ghost counts nothing in the end)
        racc[j] += f[0][j] * d;
      }
    } else {
      double below = lane_below(v[2][S_ - 1]);
      const double r = lane_above(v[0][0]);
#pragma unroll
      for (int j = 0; j < S_; j++) {
        const double up = j + 1 < S_ ? v[0][j + 1 < S_ ? j + 1 : j] : r;
        double hm = below, hp = up;
        if constexpr (kCurved) {
          hm = wl[j] * below + wl0[j] * v[0][j];
          hp = wr[j] * up + wr0[j] * v[2][j];
        }
        const double mid = v[1][j];
        below = v[2][j];
        auto step = [&](double lo, double hi, double o[3]) {
          o[0] = (P0 * hi + P1x4 * mid) * g1[j];
          o[1] = (P1 * hi + Pm * mid + P1 * lo) * g1[j];
          o[2] = (P1x4 * mid + P0 * lo) * g1[j];
        };
        double o[3], d[3];
        step(hm, hp, o);
        if constexpr (kGhost) step(hm * hl[j], hp * hr[j], d);
#pragma unroll
        for (int c = 0; c < 3; c++) {
          racc[j] += wc[c] * f[c][j] * (kGhost ? d[c] : o[c]);
          v[c][j] = o[c];
        }
      }
    }
  };

  // ---- exchange: own values to LDS, halo values back (two buffers in turn,
  // so one barrier per exchange)
  ldbl *xa = lds_row(0), *xb = lds_row(S.row_stride);
  auto exchange = [&](double (&v)[kC][S_]) {
    // the sites pass through an empty asm, so the addresses are computed here
    // and not held in registers through the steps
    int y[S_];
#pragma unroll
    for (int j = 0; j < S_; j++) {
      y[j] = x[j];
      asm volatile("" : "+v"(y[j]));
    }
    if (work) {
#pragma unroll
      for (int j = 0; j < S_; j++)
        if (real[j])
#pragma unroll
          for (int c = 0; c < kC; c++) xa[c * M + y[j]] = v[c][j];
    }
    if (nw > 1)
      lds_barrier();
    else  // one wave: its own LDS writes are in order
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    if (work) {
#pragma unroll
      for (int j = 0; j < S_; j++)
        if (halo[j])
#pragma unroll
          for (int c = 0; c < kC; c++) v[c][j] = xa[(rev[j] ? kC - 1 - c : c) * M + y[j]];
    }
    ldbl *t = xa;
    xa = xb;
    xb = t;
  };
  // kept rows: a uniform base and 32-bit lane offsets, so that no 64-bit
  // address of each lane is held through the loops
  const size_t row = (size_t)nw * 64 * S_ * kC;
  const unsigned lo = lane * S_;
  auto keep = [&](int q, const double (&v)[kC][S_]) {  // first row of segment q >= 1
    gdbl *t = hbm(S.Gf) + ((size_t)(q - 1) * row + (size_t)wave * (64 * S_ * kC));
#pragma unroll
    for (int c = 0; c < kC; c++)
#pragma unroll
      for (int j = 0; j < S_; j++) t[lo + (unsigned)(c * 64 * S_ + j)] = v[c][j];
  };
  auto fetch = [&](int q, double (&v)[kC][S_]) {
    const gdbl *t = hbm(S.Gf) + ((size_t)(q - 1) * row + (size_t)wave * (64 * S_ * kC));
#pragma unroll
    for (int c = 0; c < kC; c++)
#pragma unroll
      for (int j = 0; j < S_; j++) v[c][j] = t[lo + (unsigned)(c * 64 * S_ + j)];
  };
  auto start = [&](int b, double (&v)[kC][S_]) {  // the end segment's weight on every component
#pragma unroll
    for (int j = 0; j < S_; j++) {
      const double g = weight(b, j);
#pragma unroll
      for (int c = 0; c < kC; c++) v[c][j] = g;
    }
  };

  // ---- forward: each block in segments of up to kK rows, so a segment's
  // step weights are one block's
  double v[kC][S_];
  start(b0, v);
  load_block(b0);
  int q = 0, fresh = 0;  // segment number; steps since v's halo was exact
  for (int b = b0; b < b1; b++) {
    if (b != b0) load_block(b);
    for (int i = 0; i < S.block_n[b]; i += kK, q++) {
      const int m = S.block_n[b] - i < kK ? S.block_n[b] - i : kK;
      if (fresh + m > H) {
        exchange(v);
        fresh = 0;
      }
      fresh += m;
      if (!work) continue;
      if (q > 0) {
        step_fwd(v);
        keep(q, v);
      }
      if (m == kK) {
#pragma unroll
        for (int t = 1; t < kK; t++) step_fwd(v);
      } else {
        for (int t = 1; t < m; t++) step_fwd(v);
      }
    }
  }
  // GN over the last row, one site per thread
  if (work) {
#pragma unroll
    for (int j = 0; j < S_; j++)
      if (real[j])
#pragma unroll
        for (int c = 0; c < kC; c++) xa[c * M + x[j]] = v[c][j];
  }
  lds_barrier();
  {
    double a[kC];
#pragma unroll
    for (int c = 0; c < kC; c++) a[c] = 0.0;
    for (int i = work_tid(S); i <= MX; i += S.threads) {
      if (i < 1) continue;
      const double w = kCurved ? hbm(S.L)[i] : S.wplanar;
#pragma unroll
      for (int c = 0; c < kC; c++) a[c] += w * xa[c * M + i];
    }
    double gn = wg_sum(a[0]);
    if constexpr (kC == 3) {
      gn += 4.0 * wg_sum(a[1]);
      gn += wg_sum(a[2]);
      gn /= 6.0;
    }
    if (threadIdx.x == 0) S0.sc->GN[mo] = gn;
  }
  {  // the next exchange uses the other buffer
    ldbl *t = xa;
    xa = xb;
    xb = t;
  }

  // ---- backward with composition, segment by segment; the last row, G1
  // with the forward row still in v, first
  double next[kC][S_];  // the first row of the segment to come
  q--;
  if (work) {
    double e[kC][S_];
    start(b1 - 1, e);
#pragma unroll
    for (int j = 0; j < S_; j++) {
      racc[j] = 0.0;
#pragma unroll
      for (int c = 0; c < kC; c++) {
        if (!ghost[j]) racc[j] += (kC == 1 ? 1.0 : wc[c]) * v[c][j] * e[c][j];
        v[c][j] = e[c][j];
      }
    }
    if (q > 0)
      fetch(q, next);
    else
      start(b0, next);
  }
  fresh = 0;
  for (int b = b1 - 1; b >= b0; b--) {
    if (b != b1 - 1) load_block(b);
    const int n = S.block_n[b];
    for (int i = (n - 1) / kK * kK; i >= 0; i -= kK, q--) {
      const int left = (b == b1 - 1 ? n - 1 : n) - i;  // the last row is done
      const int m = left < kK ? left : kK;
      if (fresh + m > H) {
        exchange(v);
        fresh = 0;
      }
      fresh += m;
      if (!work) continue;
      double f[kK][kC][S_];
#pragma unroll
      for (int c = 0; c < kC; c++)
#pragma unroll
        for (int j = 0; j < S_; j++) f[0][c][j] = next[c][j];
      if (q > 1)
        fetch(q - 1, next);
      else if (q == 1)
        start(b0, next);
      auto segment = [&](auto tag) {
        if (m == kK) {
#pragma unroll
          for (int t = 1; t < kK; t++) {
#pragma unroll
            for (int c = 0; c < kC; c++)
#pragma unroll
              for (int j = 0; j < S_; j++) f[t][c][j] = f[t - 1][c][j];
            step_fwd(f[t]);
          }
#pragma unroll
          for (int t = kK - 1; t >= 0; t--) step_bwd(tag, v, f[t]);
        } else {
#pragma unroll
          for (int t = 1; t < kK - 1; t++) {
#pragma unroll
            for (int c = 0; c < kC; c++)
#pragma unroll
              for (int j = 0; j < S_; j++) f[t][c][j] = f[t - 1][c][j];
            if (t < m) step_fwd(f[t]);
          }
#pragma unroll
          for (int t = kK - 2; t >= 0; t--)
            if (t < m) step_bwd(tag, v, f[t]);
        }
      };
      if (ghosts)
        segment(std::integral_constant<bool, true>());
      else
        segment(std::integral_constant<bool, false>());
    }
    if (work) {
      gdbl *rho = hbm(S.rho) + (size_t)S.block_mm[b] * M;
#pragma unroll
      for (int j = 0; j < S_; j++) {
        if (ghost[j]) {
          // from the site's segment weight to the ghost's (both weights of a
          // curved first-order step are zero there)
          const double g = weight(b, j);
          const double to = kC == 1 && kCurved ? 0.0 : G1[(size_t)S.block_seg[b] * M + (unsigned)(p0 + j)];
          if (g != 0.0) rho[(unsigned)(p0 + j)] += racc[j] * (to / g);
        } else if (real[j]) {
          rho[(unsigned)x[j]] += racc[j];
        }
        racc[j] = 0.0;
      }
    }
  }
  __syncthreads();
}

// Whether the tiles serve molecule mo of a 1-gradient system: an unrefined
// lattice whose waves are there, for second order a simple-cubic stencil and
// no periodic boundary (set_bounds(X, Y) exchanges the two directions there,
// src/LGrad1.cpp:787-804, which no unfolded lattice does), and no weight on a surface ghost (the planar step has no separate weight for
// its missing neighbour, and second-order set_bounds pairs the two directions
// there; with the frozen segment that a surface needs the weight is zero, but
// a tagged segment's mask may not be).
template <typename Sys>
__device__ __forceinline__ bool tile_serves(const Sys &S, int mo) {
  if (S.gradients != 1 || S.fjc != 1 || !S.use_lds || tile_waves(S.M, S.mol_size[mo]) * 64 > S.threads) return false;
  if (S.mol_markov[mo] == 2 && (S.lattice_type != 0 || (S.MX > 1 && S.bx1 == S.MX))) return false;
  if (!S.surface_lo && !S.surface_hi) return true;
  bool zero = true;
  for (int b = S.mol_block_begin[mo]; b < S.mol_block_begin[mo + 1]; b++) {
    const gdbl *g = hbm(S.G1) + (size_t)S.block_seg[b] * S.M;
    if (S.surface_lo && g[0] != 0.0) zero = false;
    if (S.surface_hi && g[S.M - 1] != 0.0) zero = false;
  }
  return zero;
}

}  // namespace nscf
