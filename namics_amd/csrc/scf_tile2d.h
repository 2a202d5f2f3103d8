// First-order chains on unrefined 2-gradient lattices over many workgroups:
// up to kT2H contour steps of a lattice tile per launch.  Device code,
// included by scf_grid.hip.
#pragma once

namespace nscf {
namespace {

// A workgroup holds a tile of kT2Waves kT2S columns (x) by 64 layers (y) in
// registers: a wave owns kT2S columns, its lanes run along y.  The inner
// kT2OwnX by kT2OwnY sites are the tile's own, kT2H on every side are a halo
// of its neighbours' sites, which goes stale by one site per step, so a
// launch takes up to kT2H steps from one row in memory to the next and the
// workgroups never wait for each other.  Within a step the y neighbours come
// from the adjacent lanes (DPP) and the columns next to a wave's through LDS,
// one barrier each.
//
// What bounds a lattice of this size is its serial chain on one compute unit:
// 128 x 256 layers with the rows in HBM took 60 us per step of one workgroup.
// Steps of one launch each would pay 2.5 us of launch per step; 8 steps per
// launch pay for the halo (2048 sites computed for 768 owned) with units that
// would be idle.
constexpr int kT2S = 4, kT2Waves = 8;  // (kT2H: scf_device.h)
constexpr int kT2Threads = 64 * kT2Waves;
constexpr int kT2OwnX = kT2S * kT2Waves - 2 * kT2H, kT2OwnY = 64 - 2 * kT2H;

template <int kCtrl>
__device__ __forceinline__ double lane_shift(double v) {  // 0x138: lane i - 1, 0x130: lane i + 1
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, kCtrl, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), kCtrl, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// The layer 1..n that position p stands for when the boundaries are unfolded
// (lower ghost = layer lo, upper ghost = layer hi: a mirror or the opposite
// side), and whether it lies there reversed; 0 where it is further from the
// lattice than the halo reaches.
__device__ __forceinline__ int unfold_layer(int p, int n, int lo, int hi, bool &rev) {
  rev = false;
  if (p >= 1 && p <= n) return p;
  const bool down = p < 1;
  int steps = down ? 1 - p : p - n;
  if (steps > kT2H + 1) return 0;
  int x = down ? 1 : n;
  for (; steps > 0; steps--) {
    x += down != rev ? -1 : 1;
    if (x < 1) {
      if (lo == 1) rev = !rev;
      x = lo;
    } else if (x > n) {
      if (hi == n) rev = !rev;
      x = hi;
    }
  }
  return x;
}

struct Tile2 {
  int site[kT2S];              // lattice site of each column at this lane's layer, -1: none
  bool own[kT2S];              // this tile's own site
  double lm[kT2S], lp[kT2S];   // weights of the lower and upper column
  double C1, C2;
  int wave, lane;
  __attribute__((address_space(3))) double *edge;  // [2][waves][2][64]
  int buf;

  __device__ __forceinline__ void place(CSys &S) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ty = blockIdx.x, tx = blockIdx.y;
    const bool cyl = S.geometry != 0, sc = S.lattice_type == 0;
    C1 = sc ? 4.0 / 6.0 : 0.5;
    C2 = sc ? 1.0 / 6.0 : 0.25;
    bool ry;
    const int py = ty * kT2OwnY - kT2H + lane + 1;
    const int y = unfold_layer(py, S.MY, S.by1, S.bym, ry);
    const bool oy = lane >= kT2H && lane < kT2H + kT2OwnY && py <= S.MY;
#pragma unroll
    for (int k = 0; k < kT2S; k++) {
      const int at = wave * kT2S + k;
      const int px = tx * kT2OwnX - kT2H + at + 1;
      bool rx;
      const int x = unfold_layer(px, S.MX, S.bx1, S.bxm, rx);
      site[k] = x > 0 && y > 0 ? x * S.JX + y : -1;
      own[k] = oy && at >= kT2H && at < kT2H + kT2OwnX && px <= S.MX;
      double a = C2, b = C2;
      if (cyl && x > 0) {
        a = hbm(S.lam_m)[x * S.JX + 1];
        b = hbm(S.lam_p)[x * S.JX + 1];
      }
      lm[k] = rx ? b : a;
      lp[k] = rx ? a : b;
    }
    buf = 0;
  }
  __device__ __forceinline__ void load(const gdbl *row, double (&v)[kT2S]) const {
#pragma unroll
    for (int k = 0; k < kT2S; k++) v[k] = site[k] >= 0 ? row[(unsigned)site[k]] : 0.0;
  }
  __device__ __forceinline__ void store(gdbl *row, const double (&v)[kT2S]) const {
#pragma unroll
    for (int k = 0; k < kT2S; k++)
      if (own[k]) row[(unsigned)site[k]] = v[k];
  }
  // one step in place: the factored 9-point stencil (column sums over y, then
  // across x; LGrad2::propagate src/LGrad2.cpp:1058-1073,
  // src/LG2Planar.cpp:1085-1096), times the segment weight
  __device__ __forceinline__ void step(const double (&g1)[kT2S], double (&v)[kT2S]) {
    double q[kT2S];
#pragma unroll
    for (int k = 0; k < kT2S; k++) {
      q[k] = C1 * v[k];
      q[k] += C2 * lane_shift<0x138>(v[k]);
      q[k] += C2 * lane_shift<0x130>(v[k]);
    }
    auto *e = edge + buf * (kT2Waves * 128);
    e[wave * 128 + lane] = q[0];
    e[wave * 128 + 64 + lane] = q[kT2S - 1];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    // the outermost columns of the tile have no neighbour wave and take any
    // value: they are the first to go stale
    double qm = e[(wave > 0 ? wave - 1 : 0) * 128 + 64 + lane];
    const double qr = e[(wave < kT2Waves - 1 ? wave + 1 : wave) * 128 + lane];
    buf ^= 1;
#pragma unroll
    for (int k = 0; k < kT2S; k++) {
      const double qp = k + 1 < kT2S ? q[k + 1 < kT2S ? k + 1 : k] : qr;
      double t = C1 * q[k];
      t += lm[k] * qm;
      t += lp[k] * qp;
      v[k] = t * g1[k];
      qm = q[k];
    }
  }
};

// Forward: m steps of segment weight `seg` from a row (the chain's first
// weight, seg0 >= 0, or Gf slot src) to Gf slot dst.
__global__ void __launch_bounds__(kT2Threads) k_tile2_fwd(const DevSys *__restrict__ d, int seg0, int src, int dst,
                                                          int seg, int m) {
  __shared__ double edges[2 * kT2Waves * 128];
  CSys &S = uniform_sys(*d);
  Tile2 T;
  T.edge = (__attribute__((address_space(3))) double *)edges;
  T.place(S);
  const size_t M = S.M;
  double g1[kT2S], v[kT2S];
  T.load(hbm(S.G1) + (size_t)seg * M, g1);
  T.load(seg0 >= 0 ? hbm(S.G1) + (size_t)seg0 * M : hbm(S.Gf) + (size_t)src * M, v);
  for (int t = 0; t < m; t++) T.step(g1, v);
  T.store(hbm(S.Gf) + (size_t)dst * M, v);
}

// Backward with composition over a segment of m rows of one block: its
// forward rows are recomputed into registers from the row before them (as
// the forward pass computed them; kStart: the first of them is the chain's
// first weight, seg0, itself), then the backward rows, from Gb[bsrc] or
// (last: the segment ends the chain) from the segment weight, are composed
// with them and the last one goes to Gb[1 - bsrc].
template <bool kStart>
__global__ void __launch_bounds__(kT2Threads) k_tile2_bwd(const DevSys *__restrict__ d, int seg0, int src, int seg,
                                                          int mm, int m, int last, int bsrc) {
  __shared__ double edges[2 * kT2Waves * 128];
  CSys &S = uniform_sys(*d);
  Tile2 T;
  T.edge = (__attribute__((address_space(3))) double *)edges;
  T.place(S);
  const size_t M = S.M;
  double g1[kT2S], v[kT2S], w[kT2S], f[kT2H][kT2S], r[kT2S];
  T.load(hbm(S.G1) + (size_t)seg * M, g1);
  T.load(seg0 >= 0 ? hbm(S.G1) + (size_t)seg0 * M : hbm(S.Gf) + (size_t)src * M, w);
  if (!last) T.load(hbm(S.Gb) + (size_t)bsrc * M, v);
#pragma unroll
  for (int t = 0; t < kT2H; t++) {
    if (t < m && !(kStart && t == 0)) T.step(g1, w);
#pragma unroll
    for (int k = 0; k < kT2S; k++) f[t][k] = w[k];
  }
#pragma unroll
  for (int k = 0; k < kT2S; k++) r[k] = 0.0;
#pragma unroll
  for (int t = kT2H - 1; t >= 0; t--) {
    if (t >= m) continue;
    if (last && t == m - 1) {
#pragma unroll
      for (int k = 0; k < kT2S; k++) v[k] = g1[k];
    } else {
      T.step(g1, v);
    }
#pragma unroll
    for (int k = 0; k < kT2S; k++) r[k] += f[t][k] * v[k];
  }
  T.store(hbm(S.Gb) + (size_t)(1 - bsrc) * M, v);
  gdbl *rho = hbm(S.rho) + (size_t)mm * M;
#pragma unroll
  for (int k = 0; k < kT2S; k++)
    if (T.own[k]) rho[(unsigned)T.site[k]] += r[k];
}

// The launches of one molecule's chain (two rows or more): its blocks in
// segments of up to kT2H rows, Gf slot q the last row of segment q.  Returns
// the slot of the chain's last row.  (A first block of one row needs no
// launch: its row is the segment weight.)
struct Tile2Chain {
  struct Segment {
    int block, m;
    bool start;  // holds the chain's first row
  };
  std::vector<Segment> segs;
  const DevSys &h;
  int seg0;
  dim3 G, B;
  Tile2Chain(const DevSys &sys, int mo) : h(sys), B(kT2Threads) {
    const int b0 = h.mol_block_begin[mo], b1 = h.mol_block_begin[mo + 1];
    seg0 = h.block_seg[b0];
    for (int b = b0; b < b1; b++)
      for (int i = 0; i < h.block_n[b]; i += kT2H)
        segs.push_back({b, h.block_n[b] - i < kT2H ? h.block_n[b] - i : kT2H, b == b0 && i == 0});
    G = dim3((h.MY + kT2OwnY - 1) / kT2OwnY, (h.MX + kT2OwnX - 1) / kT2OwnX);
  }
  // whether segment q's input row is the first segment weight
  bool from_g1(size_t q) const { return q == 0 || (q == 1 && segs[0].m == 1); }
  int forward(DevSys *d, hipStream_t st) const {
    for (size_t q = 0; q < segs.size(); q++) {
      const Segment &s = segs[q];
      const int m = s.start ? s.m - 1 : s.m;
      if (m == 0) continue;
      hipLaunchKernelGGL(k_tile2_fwd, G, B, 0, st, d, from_g1(q) ? seg0 : -1, (int)q - 1, (int)q,
                         h.block_seg[s.block], m);
    }
    return (int)segs.size() - 1;
  }
  void backward(DevSys *d, hipStream_t st) const {
    int src = 0;
    for (size_t q = segs.size(); q-- > 0;) {
      const Segment &s = segs[q];
      const int seg = h.block_seg[s.block], mm = h.block_mm[s.block], last = q + 1 == segs.size();
      if (s.start)
        hipLaunchKernelGGL((k_tile2_bwd<true>), G, B, 0, st, d, seg0, 0, seg, mm, s.m, last, src);
      else
        hipLaunchKernelGGL((k_tile2_bwd<false>), G, B, 0, st, d, from_g1(q) ? seg0 : -1, (int)q - 1, seg, mm, s.m,
                           last, src);
      src = 1 - src;
    }
  }
};

}  // namespace
}  // namespace nscf
