// First-order chains of the 6-point 3-gradient stencil over many workgroups:
// up to kBoxH contour steps of a lattice tile per launch.  Device code,
// included by scf_grid.hip after scf_tile2d.h.
#pragma once

namespace nscf {
namespace {

// A workgroup holds a tile of kX x (2 waves) x 32 sites in registers: a
// thread owns the kX sites of a line along x, half a wave a line along z, so
// that the x neighbours are the thread's own registers, the z neighbours the
// adjacent lanes (DPP) and only the y neighbours go through LDS.  The inner
// sites are the tile's own, kBoxH on every side are a halo that goes stale by
// one site per step, so a launch takes up to kBoxH steps from one row in
// memory and workgroups never wait for each other.
//
// One launch per step was bound by its passes over memory and by the launch
// itself: on 96^3 sites a forward step moved 21 MB in 7.1 us and a backward
// step 35 MB in 9.2 us, plus 2.5 us between launches; on 53^3 sites a step
// took as long as its launch.  A tile reads row and weights once per kBoxH
// steps, and the rows between two checkpoints are brought back by the launch
// that composes them.  Chain of 20 segments, checkpoints every 4 rows: 381
// -> 230 us in 9 launches (from 48) on 96^3 sites, 53^3 sites 120 us.  What
// is left is the halo: 15360 sites computed for 4608 owned (FP64 issue and
// LDS about a third of a launch, its loads and start the rest).
constexpr int kBoxZ = 32, kBoxOwnZ = kBoxZ - 2 * kBoxH;  // (kBoxH: scf_box_plan.h)
constexpr int kBoxMaxWaves = 12;

// What every launch of a chain needs of its system, in the kernel's own
// arguments: read through the DevSys it took six loads one after the other.
struct BoxSys {
  int MX, MY, MZ, JX, JY;
  int px, py, pz;  // periodic along the axis, else mirrors on both sides
  int ty, tz;      // tiles along y and z
  size_t M;
  double *Gf, *Gb, *G1, *rho;
  const DevScalars *sc;  // FP32: the gauge shift of molecule mo of N segments
  int mo, N;
};

// The layer 1..n that position p stands for when the boundaries are unfolded
// (on 3-gradient lattices both ghosts are mirrors or both periodic images).
__device__ __forceinline__ int box_layer(int p, int n, int periodic) {
  const int period = periodic ? n : 2 * n;
  int q = (p - 1) % period;
  if (q < 0) q += period;
  return q < n ? q + 1 : 2 * n - q;
}

// Rows in FP64, or in FP32 with the molecule's gauge shift 
// (G1' = G1 e^c, scf_grid.hip).  FP32 is what a row
// is stored and summed in; the segment weights stay FP64 and a sum times its
// weight is rounded once, which leaves a third of the error in the densities
// that FP32 weights gave (3e-8 for 9e-8 of 20 steps on random fields).
template <typename T>
struct BoxMem;
template <>
struct BoxMem<double> {
  static __device__ __forceinline__ gdbl *gf(const BoxSys &S) { return hbm(S.Gf); }
  static __device__ __forceinline__ gdbl *gb(const BoxSys &S) { return hbm(S.Gb); }
  static __device__ __forceinline__ double shift(const BoxSys &) { return 1.0; }
  static __device__ __forceinline__ double unshift(const BoxSys &) { return 1.0; }
  static __device__ __forceinline__ double add(double rho, double f, double v, double) { return rho + f * v; }
};
template <>
struct BoxMem<float> {
  static __device__ __forceinline__ gflt *gf(const BoxSys &S) { return hbmf((float *)S.Gf); }
  static __device__ __forceinline__ gflt *gb(const BoxSys &S) { return hbmf((float *)S.Gb); }
  static __device__ __forceinline__ double shift(const BoxSys &S) { return exp(S.sc->lnshift[S.mo]); }
  static __device__ __forceinline__ double unshift(const BoxSys &S) {
    return exp(-S.sc->lnshift[S.mo] * (S.N + 1));
  }
  static __device__ __forceinline__ double add(double rho, float f, float v, double u) {
    return rho + (double)f * (double)v * u;
  }
};

template <int kCtrl>
__device__ __forceinline__ float lane_shift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF, true));
}

__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename T, int kX>
struct Box {
  typedef __attribute__((address_space(3))) T lT;
  lT *col;         // this thread's line in LDS, pitch apart in x
  int pitch;       // sites of a yz plane of the tile
  int ey, ny;      // this thread's y in the tile, the tile's lines
  int wave;
  unsigned at;     // offset of this thread's (y, z) in a lattice plane
  int xsrc;        // lane e: lattice layer of the tile's x = e
  bool own;        // (y, z) is this tile's own
  int xend;        // own x: kBoxH .. xend - 1
  int JX;

  __device__ __forceinline__ void place(const BoxSys &S, lT *lds, int waves) {
    const int lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    ny = 2 * waves;
    pitch = 64 * waves;
    ey = threadIdx.x >> 5;
    col = lds + threadIdx.x;
    JX = S.JX;
    const int own_y = ny - 2 * kBoxH;
    const int L = xcd_block_id();
    const int bz = L % S.tz, by = (L / S.tz) % S.ty, bx = L / (S.tz * S.ty);
    const int ez = lane & 31;
    const int pz = bz * kBoxOwnZ - kBoxH + ez + 1, py = by * own_y - kBoxH + ey + 1;
    const int px0 = bx * (kX - 2 * kBoxH) - kBoxH + 1;
    at = box_layer(py, S.MY, S.py) * S.JY + box_layer(pz, S.MZ, S.pz);
    own = ey >= kBoxH && ey < ny - kBoxH && py <= S.MY && ez >= kBoxH && ez < kBoxZ - kBoxH && pz <= S.MZ;
    xsrc = box_layer(px0 + (lane < kX ? lane : 0), S.MX, S.px);
    const int last = S.MX - px0 + 1;
    xend = last < kX - kBoxH ? last : kX - kBoxH;
  }
  __device__ __forceinline__ int plane(int e) const { return __builtin_amdgcn_readlane(xsrc, e) * JX; }
  template <typename Row>
  __device__ __forceinline__ void load(Row row, T (&v)[kX]) const {
#pragma unroll
    for (int e = 0; e < kX; e++) v[e] = (row + plane(e))[at];
  }
  // segment weights times a factor
  template <typename V>
  __device__ __forceinline__ void weights(const BoxSys &S, int seg, double factor, V (&g)[kX]) const {
    const gdbl *row = hbm((const double *)S.G1) + seg * S.M;
#pragma unroll
    for (int e = 0; e < kX; e++) g[e] = (V)((row + plane(e))[at] * factor);
  }
  // own sites of a row to memory
  template <typename Row>
  __device__ __forceinline__ void store(Row row, const T (&v)[kX]) const {
    if (own) {
#pragma unroll
      for (int e = kBoxH; e < kX - kBoxH; e++)
        if (e < xend) (row + plane(e))[at] = v[e];
    }
  }
  template <typename Row, typename V>
  __device__ __forceinline__ void load_own(Row row, V (&f)[kX - 2 * kBoxH]) const {
    if (own) {
#pragma unroll
      for (int e = 0; e < kX - 2 * kBoxH; e++) f[e] = (row + plane(e + kBoxH))[at];
    }
  }
  template <typename Row, typename V>
  __device__ __forceinline__ void store_own(Row row, const V (&f)[kX - 2 * kBoxH]) const {
    if (own) {
#pragma unroll
      for (int e = 0; e < kX - 2 * kBoxH; e++)
        if (e + kBoxH < xend) (row + plane(e + kBoxH))[at] = f[e];
    }
  }
  // step s of a launch in place: the sum of the six neighbours in pairs
  // (LGrad3::propagate src/LGrad3.cpp:731-743), times g, the segment weight
  // over 6.
  // The pairs make a mirrored image of a site the same number bit for bit, so
  // a row does not depend on how the steps are cut into launches.
  template <int s>
  __device__ __forceinline__ void step(const double (&g)[kX], T (&v)[kX]) const {
    tile_barrier();  // the reads of the step before
#pragma unroll
    for (int e = s + 1; e < kX - 1 - s; e++) col[e * pitch] = v[e];
    tile_barrier();
    if (2 * wave + 1 > s && 2 * wave < ny - 1 - s) {
      T below = v[s];
#pragma unroll
      for (int e = s + 1; e < kX - 1 - s; e++) {
        const T c = v[e];
        const T x = below + v[e + 1];
        const T y = col[e * pitch - 32] + col[e * pitch + 32];
        const T z = lane_shift<0x138>(c) + lane_shift<0x130>(c);
        below = c;
        v[e] = (T)((double)((x + y) + z) * g[e]);
      }
    }
  }
};

extern __shared__ __align__(16) char box_lds[];

template <typename T, int kX>
__device__ __forceinline__ void box_forward(const BoxSys &S, const Box<T, kX> &box, const BoxForward &a, T (&v)[kX],
                                            double (&g)[kX], double shift) {
  typedef BoxMem<T> Mem;
  const size_t M = S.M;
  if (a.src < 0)
    box.weights(S, a.seg0, shift, v);
  else
    box.load(Mem::gf(S) + a.src * M, v);
  box.weights(S, a.seg[0], shift * (1.0 / 6.0), g);
  if (a.slot0 >= 0) box.store(Mem::gf(S) + a.slot0 * M, v);
#define NSCF_BOX_STEP(s)                                                                 \
  if (a.n > s) {                                                                         \
    if (s > 0 && a.seg[s] != a.seg[s - (s > 0)]) box.weights(S, a.seg[s], shift * (1.0 / 6.0), g); \
    box.template step<s>(g, v);                                                          \
    if (a.slot[s] >= 0) box.store(Mem::gf(S) + a.slot[s] * M, v);                        \
  }
  NSCF_BOX_STEP(0)
  NSCF_BOX_STEP(1)
  NSCF_BOX_STEP(2)
  NSCF_BOX_STEP(3)
#undef NSCF_BOX_STEP
}

template <typename T, int kX>
__global__ void __launch_bounds__(64 * kBoxMaxWaves) k_box_fwd(BoxSys S, BoxForward a, int waves) {
  Box<T, kX> box;
  box.place(S, (typename Box<T, kX>::lT *)box_lds, waves);
  T v[kX];
  double g[kX];
  box_forward<T, kX>(S, box, a, v, g, BoxMem<T>::shift(S));
}

// The backward rows with the composition rho += Gf Gb of each, after the
// forward steps whose rows they compose: a thread reads back the sites that
// it wrote itself.
template <typename T, int kX>
__global__ void __launch_bounds__(64 * kBoxMaxWaves) k_box_bwd(BoxSys S, BoxRun a, int waves) {
  typedef BoxMem<T> Mem;
  constexpr int kOwn = kX - 2 * kBoxH;
  const size_t M = S.M;
  Box<T, kX> box;
  box.place(S, (typename Box<T, kX>::lT *)box_lds, waves);
  T v[kX], f[kOwn] = {};
  double g[kX], rho[kOwn] = {};
  const double shift = Mem::shift(S), u = Mem::unshift(S);
  if (a.f.n > 0) box_forward<T, kX>(S, box, a.f, v, g, shift);
  if (a.src < 0)
    box.weights(S, a.seg0, shift, v);
  else
    box.load(Mem::gb(S) + a.src * M, v);
  if (a.n > 0) box.weights(S, a.seg[0], shift * (1.0 / 6.0), g);
  int mm = a.slot0 >= 0 ? a.mm0 : a.mm[0];
  box.load_own(hbm(S.rho) + mm * M, rho);
  if (a.slot0 >= 0) {
    box.load_own(Mem::gf(S) + a.slot0 * M, f);
#pragma unroll
    for (int e = 0; e < kOwn; e++) rho[e] = Mem::add(rho[e], f[e], v[e + kBoxH], u);
  }
#define NSCF_BOX_STEP(s)                                                             \
  if (a.n > s) {                                                                     \
    if (s > 0 && a.seg[s] != a.seg[s - (s > 0)]) box.weights(S, a.seg[s], shift * (1.0 / 6.0), g); \
    if (a.mm[s] != mm) {                                                             \
      box.store_own(hbm(S.rho) + mm * M, rho);                                       \
      mm = a.mm[s];                                                                  \
      box.load_own(hbm(S.rho) + mm * M, rho);                                        \
    }                                                                                \
    box.load_own(Mem::gf(S) + a.slot[s] * M, f);                                     \
    box.template step<s>(g, v);                                                      \
    _Pragma("unroll") for (int e = 0; e < kOwn; e++) rho[e] = Mem::add(rho[e], f[e], v[e + kBoxH], u); \
  }
  NSCF_BOX_STEP(0)
  NSCF_BOX_STEP(1)
  NSCF_BOX_STEP(2)
  NSCF_BOX_STEP(3)
#undef NSCF_BOX_STEP
  box.store_own(hbm(S.rho) + mm * M, rho);
  box.store(Mem::gb(S) + a.dst * M, v);
}

// The tile shape of a lattice: rounds of tiles over the compute units (one
// tile each) times the sites a tile computes, the least.  Solves of 12
// iterations: on 96^3 sites x = 20, 12 waves 7.7 ms (the rule's choice),
// 24, 12 9.2, 16, 12 8.9, 12, 8 8.3; on 53^3 x = 16, 8 waves 3.41 (its
// choice), 12, 12 3.38, 20, 12 4.4, 24, 12 5.6.
struct BoxShape {
  int kx, waves, tiles;
  explicit BoxShape(const DevSys &h) {
    long best = 0;
    for (int x : {12, 16, 20, 24})
      for (int w : {8, 12}) {
        const int oy = 2 * w - 2 * kBoxH, ox = x - 2 * kBoxH;
        const int n = ((h.MX + ox - 1) / ox) * ((h.MY + oy - 1) / oy) * ((h.MZ + kBoxOwnZ - 1) / kBoxOwnZ);
        const long cost = (long)((n + 255) / 256) * x * w;
        if (best && cost >= best) continue;
        best = cost;
        kx = x;
        waves = w;
        tiles = n;
      }
  }
};

template <typename T, int kX>
hipError_t box_launch(const BoxShape &shape, const BoxSys &S, const BoxForward *f, const BoxRun *b, hipStream_t st) {
  const size_t lds = (size_t)kX * 64 * shape.waves * sizeof(T);
  const void *k = f ? (const void *)k_box_fwd<T, kX> : (const void *)k_box_bwd<T, kX>;
  const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  const dim3 G(shape.tiles), B(64 * shape.waves);
  if (f)
    hipLaunchKernelGGL((k_box_fwd<T, kX>), G, B, lds, st, S, *f, shape.waves);
  else
    hipLaunchKernelGGL((k_box_bwd<T, kX>), G, B, lds, st, S, *b, shape.waves);
  return hipSuccess;
}

template <typename T>
hipError_t box_launch(const BoxShape &s, const BoxSys &S, const BoxForward *f, const BoxRun *b, hipStream_t st) {
  switch (s.kx) {
    case 12: return box_launch<T, 12>(s, S, f, b, st);
    case 16: return box_launch<T, 16>(s, S, f, b, st);
    case 20: return box_launch<T, 20>(s, S, f, b, st);
    default: return box_launch<T, 24>(s, S, f, b, st);
  }
}

// The chain of molecule mo in launches of up to kBoxH rows.
struct BoxChain {
  const BoxShape shape;
  BoxSchedule plan;
  bool fp32;
  BoxSys S;
  BoxChain(const DevSys &h, int mo, bool f32) : shape(h), plan(h.mol_N[mo], h.ckpt), fp32(f32) {
    for (int b = h.mol_block_begin[mo]; b < h.mol_block_begin[mo + 1]; b++) {
      plan.seg.insert(plan.seg.end(), h.block_n[b], h.block_seg[b]);
      plan.mm.insert(plan.mm.end(), h.block_n[b], h.block_mm[b]);
    }
    const int own_y = 2 * shape.waves - 2 * kBoxH;
    S = {h.MX, h.MY, h.MZ, h.JX, h.JY,
         h.bx1 != 1, h.by1 != 1, h.bz1 != 1,
         (h.MY + own_y - 1) / own_y, (h.MZ + kBoxOwnZ - 1) / kBoxOwnZ, (size_t)h.M,
         h.Gf, h.Gb, h.G1, h.rho, h.sc, mo, h.mol_N[mo]};
  }
  // The whole chain; gn(slot) launches the sum over the last row while it is
  // held there.
  template <typename Gn>
  hipError_t run(hipStream_t st, Gn gn) const {
    return (hipError_t)plan.run(
        [&](const BoxForward *f, const BoxRun *b) -> int {
          return fp32 ? box_launch<float>(shape, S, f, b, st) : box_launch<double>(shape, S, f, b, st);
        },
        [&] { gn(plan.loc(plan.N - 1)); });
  }
};

}  // namespace
}  // namespace nscf
