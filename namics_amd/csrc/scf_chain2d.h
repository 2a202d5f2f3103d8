// First-order chains on unrefined 2-gradient lattices in one workgroup: the
// whole lattice in registers.  Device code, included by scf_fused.hip after
// its LDS helpers and scf_chain1d.h.
#pragma once

namespace nscf {

// A wave owns SX columns (x), its lanes run along y with YP consecutive
// layers each (SX YP = 8 sites per thread), so the y neighbours come from the
// lane itself or the adjacent lanes (DPP) and only the column sums of a
// wave's two outer columns go through LDS: 64 bytes per thread and step with
// one barrier, where keeping the row in LDS moved 240 (64 x 128 layers: 1.7
// us per step, bound by that traffic; strips remain for the FP32 chains and for
// shapes that leave too many lanes idle, registers_faster in scf_api.hip).  Any number of layers fits that has
// the lanes and waves: MY <= 64 YP, MX <= 16 SX.  (kFull: every lane and
// column is inside the lattice.)
//
// The step is the factored 9-point stencil (column sums over y, then across
// x; LGrad2::propagate src/LGrad2.cpp:1058-1073, LG2Planar::propagate
// src/LG2Planar.cpp:1085-1096), its sums in the order of strip_step.
//
// End-point rows in memory are MX columns of MY (rounded up to YP) layers.
// With checkpoints of interval K the forward pass keeps rows 0, K, 2K, ...;
// the backward pass recomputes the others: up to K = 4 on chip (the first of
// a segment's rows is kept in LDS, the later ones start from it, the base row
// is read again), beyond that through a buffer of K - 1 rows in memory.  With
// one system per CU the rows of 256 systems saturate HBM, and what the
// interval saves there is worth the steps.
//
// Measured on one MI355X, chains per evaluation: 64 x 128, N = 200, one
// system 0.68 -> 0.44 ms (1.1 us per step, half of it the 72 vector
// instructions of 4 waves per SIMD, the rest the LDS exchange and its
// barrier); 256 systems 1.04 (interval 2) -> 0.65 ms (interval 3); 43 x 101,
// N = 120, which the strips cannot divide, 1.34 -> 0.26 ms.
template <int YP, bool kFull>
struct Wave2 {
  static constexpr int SX = kWave2Sites / YP;
  typedef double Sites[SX][YP];

  int MX, MY, JX, lane, wave, nw, cols;  // cols: columns of this wave inside the lattice
  bool work, on;                         // this wave, this lane holds sites
  double Cy[YP];                         // weight of a site's own value in its column sum
  int top_lane, top_j;                   // of the uppermost layer
  bool py, px;                           // periodic along y, x
  double C1, C2;
  double Cx[SX], lm[SX], lp[SX];         // weights of a column's own sum and of its neighbours'
  unsigned site0, row0;                  // of (k, j) = (0, 0): in lattice arrays, in a stored row
  unsigned ystride;                      // stored layers per column
  size_t row;                            // doubles of a stored row
  ldbl *edge;                            // [2][nw][2][64 YP] column sums
  ldbl *own;                             // [8][1024] values of this thread (recomputed row)
  int buf;

  __device__ __forceinline__ void place(CSys &S) {
    MX = S.MX;
    MY = S.MY;
    JX = S.JX;
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    nw = (MX + SX - 1) / SX;
    work = wave < nw;
    cols = kFull || MX - wave * SX > SX ? SX : MX - wave * SX;
    const int lanes = (MY + YP - 1) / YP;
    on = work && (kFull || lane < lanes);
    top_lane = (MY - 1) / YP;
    top_j = (MY - 1) % YP;
    py = S.by1 != 1;  // (one layer: its opposite side is itself)
    px = S.bx1 != 1;
    const bool sc = S.lattice_type == 0;
    C1 = sc ? 4.0 / 6.0 : 0.5;
    C2 = sc ? 1.0 / 6.0 : 0.25;
    // past a mirror lies the site itself; the neighbour read there (an edge
    // lane's missing one, or a site beyond the lattice, which stays 0) is 0
#pragma unroll
    for (int j = 0; j < YP; j++) {
      Cy[j] = C1;
      if (!py && lane == 0 && j == 0) Cy[j] += C2;
      if (!py && lane == top_lane && j == top_j) Cy[j] += C2;
    }
    const int x0 = wave * SX + 1;
#pragma unroll
    for (int k = 0; k < SX; k++) {
      lm[k] = lp[k] = C2;
      if (S.geometry != 0 && work && k < cols) {
        typedef const __attribute__((address_space(4))) double kdbl;
        lm[k] = ((kdbl *)S.lam_m)[(x0 + k) * JX + 1];
        lp[k] = ((kdbl *)S.lam_p)[(x0 + k) * JX + 1];
      }
      // past a mirror lies the column itself; where there is none, nothing
      Cx[k] = C1;
      if (!px && x0 + k == 1) {
        Cx[k] += lm[k];
        lm[k] = 0.0;
      }
      if (!px && x0 + k == MX) {
        Cx[k] += lp[k];
        lp[k] = 0.0;
      }
    }
    ystride = lanes * YP;
    row = (size_t)MX * ystride;
    const unsigned l = on ? lane : 0;
    site0 = (work ? x0 : 1) * JX + l * YP + 1;
    row0 = (work ? x0 - 1 : 0) * ystride + l * YP;
    edge = lds_row(0);
    own = lds_row(2 * nw * 128 * YP) + (int)threadIdx.x;
    buf = 0;
  }
  // lattice array -> sites (0 outside the lattice, where nothing ever grows).
  // Here and below a column's address is a uniform base plus one 32-bit lane
  // offset for all columns: 64-bit addresses of each would be hoisted out of
  // the step loops and spill there.
  __device__ __forceinline__ void load_sites(const gdbl *a, Sites &v) const {
#pragma unroll
    for (int k = 0; k < SX; k++) {
      const gdbl *c = a + k * JX;
#pragma unroll
      for (int j = 0; j < YP; j++) v[k][j] = on && k < cols && lane * YP + j < MY ? c[site0 + (unsigned)j] : 0.0;
    }
  }
  // (two forms, so that a full wave's four accesses are not four branches)
  __device__ __forceinline__ void load_row(const gdbl *r, Sites &v) const {
    if (!on) return;
    auto column = [&](int k) {
      const gdbl *c = r + k * ystride;
#pragma unroll
      for (int j = 0; j < YP; j++) v[k][j] = c[row0 + (unsigned)j];
    };
    if (cols == SX) {
#pragma unroll
      for (int k = 0; k < SX; k++) column(k);
    } else {
#pragma unroll
      for (int k = 0; k < SX; k++)
        if (k < cols) column(k);
    }
  }
  __device__ __forceinline__ void store_row(gdbl *r, const Sites &v) const {
    if (!on) return;
    auto column = [&](int k) {
      gdbl *c = r + k * ystride;
#pragma unroll
      for (int j = 0; j < YP; j++) c[row0 + (unsigned)j] = v[k][j];
    };
    if (cols == SX) {
#pragma unroll
      for (int k = 0; k < SX; k++) column(k);
    } else {
#pragma unroll
      for (int k = 0; k < SX; k++)
        if (k < cols) column(k);
    }
  }
  __device__ __forceinline__ void keep_own(const Sites &v) const {
#pragma unroll
    for (int k = 0; k < SX; k++)
#pragma unroll
      for (int j = 0; j < YP; j++) own[(k * YP + j) * 1024] = v[k][j];
  }
  __device__ __forceinline__ void load_own(Sites &v) const {
#pragma unroll
    for (int k = 0; k < SX; k++)
#pragma unroll
      for (int j = 0; j < YP; j++) v[k][j] = own[(k * YP + j) * 1024];
  }

  // YP column sums of a lane to and from LDS, 16 bytes at a time (8-byte
  // accesses at a stride of 16 would meet in the banks)
  typedef double d2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) d2 ld2;
  static __device__ __forceinline__ void put(ldbl *e, const double (&a)[YP]) {
    if constexpr (YP == 1) {
      e[0] = a[0];
    } else {
#pragma unroll
      for (int j = 0; j < YP; j += 2) *(ld2 *)(e + j) = d2{a[j], a[j + 1 < YP ? j + 1 : j]};
    }
  }
  static __device__ __forceinline__ void get(const ldbl *e, double (&a)[YP]) {
    if constexpr (YP == 1) {
      a[0] = e[0];
    } else {
#pragma unroll
      for (int j = 0; j < YP; j += 2) {
        const d2 t = *(const ld2 *)(e + j);
        a[j] = t.x;
        a[j + 1 < YP ? j + 1 : j] = t.y;
      }
    }
  }

  // one step in place (every wave of the workgroup calls it).  Written with
  // explicit fma, so that a row recomputed in the backward pass has the bits
  // of the forward one.
  __device__ __forceinline__ void step(const Sites &g1, Sites &v) {
    Sites q;
    auto across = [&](int k, int j, double qm, double qp) {
      const double t = __builtin_fma(lp[k], qp, __builtin_fma(lm[k], qm, Cx[k] * q[k][j]));
      v[k][j] = t * g1[k][j];
    };
    if (work) {
#pragma unroll
      for (int k = 0; k < SX; k++) {
        const double dn = lane_below(v[k][YP - 1]), up = lane_above(v[k][0]);
#pragma unroll
        for (int j = 0; j < YP; j++) {
          const double b = j > 0 ? v[k][j > 0 ? j - 1 : 0] : dn;
          const double a = j < YP - 1 ? v[k][j < YP - 1 ? j + 1 : j] : up;
          q[k][j] = __builtin_fma(C2, a, __builtin_fma(C2, b, Cy[j] * v[k][j]));
        }
      }
      if (py) {  // the opposite side's values, where the neighbour read was 0
#pragma unroll
        for (int k = 0; k < SX; k++) {
          double t = v[k][YP - 1];
#pragma unroll
          for (int j = 0; j < YP - 1; j++)
            if (j == top_j) t = v[k][j];
          const double lo = readlane_f64(t, top_lane), hi = readlane_f64(v[k][0], 0);
          q[k][0] = __builtin_fma(C2, lane == 0 ? lo : 0.0, q[k][0]);
#pragma unroll
          for (int j = 0; j < YP; j++)
            if (j == top_j) q[k][j] = __builtin_fma(C2, lane == top_lane ? hi : 0.0, q[k][j]);
        }
      }
      ldbl *e = edge + (buf * nw + wave) * (128 * YP) + lane * YP;
      put(e, q[0]);
      put(e + 64 * YP, q[SX - 1]);
      if (px && cols < SX) {  // the last column of a periodic lattice is an inner one here
#pragma unroll
        for (int k = 0; k < SX - 1; k++)
          if (k == cols - 1) put(e + 64 * YP, q[k]);
      }
      // the inner columns while the outer ones travel
#pragma unroll
      for (int k = 1; k < SX - 1; k++)
#pragma unroll
        for (int j = 0; j < YP; j++) across(k, j, q[k - 1][j], q[k + 1][j]);
    }
    lds_barrier();
    if (work) {
      const ldbl *e = edge + buf * nw * (128 * YP) + lane * YP;
      // slots of the columns below and above this wave's (any at a mirror,
      // where their weight is 0)
      const int below = wave > 0 ? 2 * (wave - 1) + 1 : 2 * (nw - 1) + 1;
      const int above = wave < nw - 1 ? 2 * (wave + 1) : 0;
      double qm[YP], qr[YP];
      get(e + below * (64 * YP), qm);
      get(e + above * (64 * YP), qr);
#pragma unroll
      for (int j = 0; j < YP; j++) {
        if constexpr (SX > 1) {
          across(0, j, qm[j], q[SX > 1 ? 1 : 0][j]);
          across(SX - 1, j, q[SX > 1 ? SX - 2 : 0][j], qr[j]);
        } else {
          across(0, j, qm[j], qr[j]);
        }
      }
      if (px && cols < SX) {  // ... and its upper neighbour the first column
#pragma unroll
        for (int k = 0; k < SX - 1; k++)
          if (k == cols - 1)
#pragma unroll
            for (int j = 0; j < YP; j++) v[k][j] = __builtin_fma(lp[k] * qr[j], g1[k][j], v[k][j]);
      }
    }
    buf ^= 1;
  }
};

// The block that holds a row of the chain.
template <typename Sys>
__device__ __forceinline__ int block_of_row(const Sys &S, int b, int r) {
  int n = S.block_n[b];
  while (r >= n) n += S.block_n[++b];
  return b;
}

// Backward pass with composition.  kBuffer: rows between checkpoints through
// memory (K > 4, or no LDS for a row); else at most 4 rows per checkpoint.
template <int YP, bool kFull, bool kBuffer>
__device__ __noinline__ void wave2_backward(const DevSys &S0, int mo) {
  typedef Wave2<YP, kFull> W2;
  constexpr int SX = W2::SX;
  CSys &S = uniform_sys(S0);
  mo = __builtin_amdgcn_readfirstlane(mo);
  W2 W;
  W.place(S);
  const int b0 = S.mol_block_begin[mo], b1 = S.mol_block_begin[mo + 1], N = S.mol_N[mo];
  const int K = S.ckpt > 1 ? S.ckpt : 1;
  const size_t M = S.M;
  const gdbl *G1 = hbm(S.G1);
  gdbl *Gf = hbm(S.Gf);
  gdbl *Bf = Gf + (size_t)((N + K - 1) / K) * W.row;  // kBuffer: rows base + 1 .. base + K - 1
  typename W2::Sites g1, v, w, racc;
  int b = b1 - 1, loaded = -1;
  auto weights = [&](int bb) {
    if (loaded == bb) return;
    W.load_sites(G1 + (size_t)S.block_seg[bb] * M, g1);
    loaded = bb;
  };
  auto forward = [&](int r) {  // w: row r - 1 -> row r
    weights(block_of_row(S, b0, r));
    W.step(g1, w);
  };
  auto flush = [&](int bb) {
    gdbl *rho = hbm(S.rho) + (size_t)S.block_mm[bb] * M;
#pragma unroll
    for (int k = 0; k < SX; k++) {
      gdbl *c = rho + k * W.JX;
#pragma unroll
      for (int j = 0; j < YP; j++) {
        if (W.on && k < W.cols && W.lane * YP + j < W.MY) c[W.site0 + (unsigned)j] += racc[k][j];
        racc[k][j] = 0.0;
      }
    }
  };
#pragma unroll
  for (int k = 0; k < SX; k++)
#pragma unroll
    for (int j = 0; j < YP; j++) racc[k][j] = w[k][j] = 0.0;
  int bstart = N - S.block_n[b], n = (N - 1) % K, seg = (N - 1) / K;  // row = seg K + n
  bool top = true;                                                      // of its segment: w holds the base row
  W.load_row(Gf + (size_t)seg * W.row, w);
  weights(b);
#pragma unroll
  for (int k = 0; k < SX; k++)
#pragma unroll
    for (int j = 0; j < YP; j++) v[k][j] = g1[k][j];
  for (int r = N - 1;; r--) {
    // the loads into w, issued at the end of the row before, have the
    // backward step to arrive in
    if (r < bstart) {
      flush(b);
      b--;
      bstart -= S.block_n[b];
    }
    if (r < N - 1) {
      weights(b);
      W.step(g1, v);
    }
    if constexpr (kBuffer) {
      if (top)
        for (int t = 1; t <= n; t++) {
          forward(r - n + t);
          if (t < n) W.store_row(Bf + (size_t)(t - 1) * W.row, w);
        }
    } else {
      int t = 1;
      if (!top && n > 0) {
        W.load_own(w);
        t = 2;
      }
      for (; t <= n; t++) {
        forward(r - n + t);
        if (t == 1 && n > 1) W.keep_own(w);
      }
    }
#pragma unroll
    for (int k = 0; k < SX; k++)
#pragma unroll
      for (int j = 0; j < YP; j++) racc[k][j] += w[k][j] * v[k][j];
    if (r == 0) break;
    top = n == 0;
    if (top) {
      seg--;
      n = K;
    }
    n--;
    if (top || n == 0)
      W.load_row(Gf + (size_t)seg * W.row, w);
    else if constexpr (kBuffer)
      W.load_row(Bf + (size_t)(n - 1) * W.row, w);
  }
  flush(b);
}

template <int YP, bool kFull>
__device__ __noinline__ void chain2d_wave(const DevSys &S0, int mo) {
  typedef Wave2<YP, kFull> W2;
  constexpr int SX = W2::SX;
  CSys &S = uniform_sys(S0);
  mo = __builtin_amdgcn_readfirstlane(mo);
  W2 W;
  W.place(S);
  const int b0 = S.mol_block_begin[mo], b1 = S.mol_block_begin[mo + 1];
  const int K = S.ckpt > 1 ? S.ckpt : 1;
  const size_t M = S.M;
  const gdbl *G1 = hbm(S.G1);
  gdbl *next = hbm(S.Gf);
  typename W2::Sites g1, v;
  W.load_sites(G1 + (size_t)S.block_seg[b0] * M, g1);
#pragma unroll
  for (int k = 0; k < SX; k++)
#pragma unroll
    for (int j = 0; j < YP; j++) v[k][j] = g1[k][j];
  W.store_row(next, v);
  next += W.row;
  int left = K;  // steps to the next kept row
  for (int b = b0; b < b1; b++) {
    if (b != b0) W.load_sites(G1 + (size_t)S.block_seg[b] * M, g1);
    for (int i = b == b0 ? 1 : 0; i < S.block_n[b]; i++) {
      W.step(g1, v);
      if (--left == 0) {
        W.store_row(next, v);
        next += W.row;
        left = K;
      }
    }
  }
  double acc = 0.0;
  {
    const gdbl *L = hbm(S.L);
    const bool cyl = S.geometry != 0;
#pragma unroll
    for (int k = 0; k < SX; k++)
#pragma unroll
      for (int j = 0; j < YP; j++)
        if (W.on && k < W.cols && W.lane * YP + j < W.MY)
          acc += (cyl ? L[W.site0 + (unsigned)(k * W.JX + j)] : 1.0) * v[k][j];
  }
  const double gn = wg_sum(acc);
  if (threadIdx.x == 0) S0.sc->GN[mo] = gn;
  if (K > 4 || (K > 2 && !S.wave2_own))
    wave2_backward<YP, kFull, true>(S0, mo);
  else
    wave2_backward<YP, kFull, false>(S0, mo);
  __syncthreads();
}

// (kFull spares the tests of lanes and columns: N = 200, per evaluation, 32 x 64
// layers 409 -> 371 us, 64 x 128 769 -> 714, 32 x 256 814 -> 787)
template <int YP>
__device__ __forceinline__ void chain_wave2_select(const DevSys &S, int mo) {
  if (S.MY == 64 * YP && S.MX % (kWave2Sites / YP) == 0)
    chain2d_wave<YP, true>(S, mo);
  else
    chain2d_wave<YP, false>(S, mo);
}

__device__ __forceinline__ void chain_wave2(const DevSys &S, int mo) {
  if (S.wave2 == 1)
    chain_wave2_select<1>(S, mo);
  else if (S.wave2 == 2)
    chain_wave2_select<2>(S, mo);
  else
    chain_wave2_select<4>(S, mo);
}

}  // namespace nscf
