// pdem_mixed.hpp -- mixed-precision state-based bond kernels (PDEM_PREC_MIXED).
//
// Bond arithmetic in FP32, sums in FP64: the dilation theta and the weighted
// volume stay FP64 (cancellation), bond forces are summed in FP32 over blocks
// of KB = 8 bonds and the blocks in FP64, and the node update stays FP64.
//
// Work unit: a tile = up to TILE_NODES consecutive nodes of one particle.
// Horizons never cross particles, so a tile's neighbors lie in a window of
// node ids [ws, we) inside its particle.  LDS tiles (the window fits) stage
// the window once per workgroup (three records of 16 bytes per node, see
// Win) and every bond reads LDS; the remaining
// tiles (particles whose numbering spreads neighbors over more ids than the
// window holds) gather from HBM through the caches: a separate
// instantiation, launched on a second stream beside the LDS tiles.
//
// Neighbor ids are 16-bit, stored in blocks of KB = 8 per lane: one 16-byte
// load yields a lane's next 8 ids and the block loop is unrolled so each id is
// a compile-time lane of the block.  In models of few different meshes the
// bond's constant weight (its reference geometry: r J(r) V_j^c) lies beside
// each id, so the loops evaluate only what moves; models of many evaluate the
// weights (GEOM_MIN_ENTRIES), and so do HBM tiles.
//
// Lists are shared: the particles of a model are mostly scaled and turned
// copies of a few meshes, whose tiles then have the same relative ids and,
// up to the particle's scale h V, the same weights.  Set-up finds such tiles
// (by hash, then by comparing every entry) and stores one list for all of
// them.  512-instance ensemble: 17167 particles, 78 lists of 0.54M entries (3 MB
// with the weights, which stay in L2).  Packing of 2000 spheres, 1.4e8 bonds:
// 101 lists of 7.3M entries (15 MB of ids), nearly all of them of one sphere
// each, whose bonds as long as the horizon fall on either side of it by the
// rounding of its turn; that is too many to read weights, and its tiles
// evaluate them.  A tile whose list matches no other keeps its own.
//
// Threads take nodes in slot order: inside every LDS tile the nodes are ordered
// by their number of 4-bond half blocks (most first, node id second), so the
// 64 lanes of a wavefront run lists of about the same length (a wavefront
// runs as long as its longest list; surface nodes have far fewer bonds than
// interior ones).  The lists are laid out by slot; node data, bond bits and
// results stay indexed by node.
//
// FMA contraction is allowed inside these kernels only (the FP64 parity
// kernels are built without it).
//
// The stretch uses the cancellation-free form
//   |xi + eta| - |xi| = (2 xi.eta + eta.eta) / (|xi + eta| + |xi|)
// so FP32 keeps ~1e-7 relative accuracy at small strains.
#pragma once
#include <type_traits>

#include "pdem_kernels.hpp"

namespace pdem {

constexpr int TILE_NODES = 1024;
constexpr int LDS_NODES = 1280;   // window of up to 1280 nodes, ~61 KB of LDS per workgroup
// Window classes: a launch whose LDS windows all hold at most LDS_SMALL nodes
// uses the small instantiation (~19 KB of LDS per workgroup, so small particles
// do not hold LDS sized for the largest window and more workgroups fit a CU).
constexpr int LDS_SMALL = 384;
// Windows of up to LDS_MID nodes leave room for three workgroups on a CU:
// there the fused kernel runs 512 threads where 1024 are asked for, two nodes
// a thread (24 wavefronts and up to 85 VGPRs instead of 32 and 64, no spills;
// 2000 spheres of 1021 nodes: 0.541 to 0.516 ms per step).
constexpr int LDS_MID = 1120;
constexpr int KB = 8;             // neighbor ids per 16-byte block
// HBM tiles (a meshed wall, a particle of many nodes) wait on gathers.  A tile
// goes to several workgroups of HBM_TPB threads, an eighth of the tiles to each
// XCD (see hbm_tile), whose L2 then holds a particle's data once.  Bonds are
// gathered 8 at a time, and their weights evaluated: read from the lists, they
// would be three times the bytes that pass through the caches (the Gaussian
// influence function's are read).  In models of up to HBM_LPN8_NODES nodes in
// such tiles, a node's list is dealt to 8 lanes, for lack of wavefronts; above,
// a lane each, so that neighboring lanes gather neighboring nodes.  For that
// the nodes keep their order, unless it is an arbitrary one (lists that span
// more than 3/4 of the particle), where lists of equal length go together.
// Both passes, us: without lanes, a workgroup of 1024 a tile / 8 lanes, weights
// read, tiles dealt to all XCDs / now; 8 lanes and one at the line:
//   sphere of 9.9k nodes              286    94    87
//   4 of 9.9k                         302   177   130 (one lane 204)
//   10 of 9.9k                        342   377   209 (8 lanes 245)
//   10 of 40k                        1005  1640   640
//   40 of 40k                        4600  6400  2247
//   20 disks of 40k                   323   727   292
//   10 spheres of 9.9k, any order     916   650   502
//   300 of 2.5k, any order           1700  4460  1740
constexpr int HBM_TPB = 256;
constexpr int64_t HBM_LPN8_NODES = 1 << 16;
// waves per SIMD the bond kernels are compiled for (at most 64 VGPRs): two
// 1024-thread workgroups per CU, so one stages its window while the other computes
constexpr int MIXED_WAVES_PER_SIMD = 8;
// HBM tiles, whose positions are FP64 and which take 8 bonds at once: first and
// second pass (at 8 the registers spill: 10 spheres of 40k nodes 807 us for both
// passes, 640 now)
constexpr int HBM_WAVES_PER_SIMD = 4, HBM_WAVES2_PER_SIMD = 6;

struct DevTile {
  int ts, te;     // nodes [ts, te)
  int ws, we;     // neighbor window [ws, we)
  int pid;
  int lds;        // window staged in LDS; 2: also closed (the tile is its whole particle)
  // the tile's list: thread slot q runs node ts + (lnode[node + q] & 0xffff)
  // with lnode[node + q] >> 16 bonds, named by col16 from element
  // data + lslice[slice + q / 64] + (q % 64) * KB on: entry k at
  // (k / KB) * 64 * KB + k % KB beyond it.  An entry is the byte offset
  // 16 (j - ws) of the neighbor's LDS records (LDS tiles, padded to whole
  // blocks with 16 (we - ws)) or j - glob_start (HBM tiles, padded with 0).
  // The weights 2 r J(r) V_j^c / particle_scale (0 in the padding) lie in
  // half blocks: wgt[data + lslice + (k / 4) * 64 * 4 + (q % 64) * 4 + k % 4].
  int node, slice;
  int64_t data;
};

// constants of a particle (set-up): particle_scale and its reciprocal, the
// largest component of the reference positions relative to the first node's
// (rounded up)
struct PartConst {
  double scale, inv_scale;
  float xmax;
};

struct MixedArgs {
  const PartConst* part;  // [np]
  const DevTile* tiles;   // closed LDS tiles, then open LDS tiles, then HBM tiles
  int ntiles_closed, ntiles_lds, ntiles_hbm;
  int hbm_lpn, hbm_split; // HBM tiles: lanes per node, workgroups per tile
  int small;              // every LDS window holds at most LDS_SMALL nodes
  int mid;                // every LDS window holds at most LDS_MID nodes
  // the lists (see DevTile)
  const uint32_t* lnode;
  const int* lslice;
  const uint16_t* col16;
  const float* wgt;
  // LDS tiles evaluate the weights from the reference positions instead of
  // reading them (lists too many to stay in cache)
  int geom;
  const float* fa;        // per node 2 alpha particle_scale, alpha = 15 G / m (constant, from set-up)
  float* fb;              // per node b particle_scale, b = theta ((3K/m) - alpha / 3), of the open tiles
  // particles with open LDS tiles: particle_max over the particle, for the
  // fixed-point steps of their windows
  const int* open_pids;
  int n_open_pids;
  float2* pmax;           // [np]
};

// The bond weights are read from the lists while the lists of the LDS tiles
// hold at most this many entries (6 bytes each; an XCD's L2 holds 4 MB) and
// evaluated from the reference positions beyond it, where their lists would
// come from HBM in both passes (constant and linear influence functions; the
// Gaussian one costs an exponential, so its weights are always read).  Lists
// that read none have none stored (has_weights).
// Measured with 1 / 16 / 64 / 256 lists of equal use and one for each particle,
// step in us, read and evaluated: packing of 2000 spheres of 1021 nodes (76k
// entries each) 478, 499, 521, 562, 645 against 486, 488, 490, 499, 518;
// 512-instance ensemble of particles of up to 367 nodes (12k entries)
// 493, 494, 504, 522, 574 against 510, 508, 513, 513, 520.
constexpr int64_t GEOM_MIN_ENTRIES = 1 << 21;

// the particle's scale h V(first node), by which the weights are divided: the
// copies of one mesh then have equal weights, and weights times alpha or b
// are of moderate size in any unit
__device__ __forceinline__ double particle_scale(const DS& s, const DevParticle& p) {
  const double c = p.h * s.vol[p.glob_start];
  return c > 1e-300 ? c : 1.;
}

// keeps the work of one group of bonds apart from the next: without it the
// compiler gathers the loads of a whole block first and runs out of registers
__device__ __forceinline__ void pin(float (&f)[3], float& z) {
  asm volatile("" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(z)::"memory");
}
// a value that is the same in every lane, kept in a scalar register
__device__ __forceinline__ float uniform(float x) {
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
}
__device__ __forceinline__ float rcpf(float x) { return __builtin_amdgcn_rcpf(x); }
// hardware reciprocal square root (1 ulp, no denormal rescaling): bond lengths
// squared are far from the FP32 denormal range.  It yields both
// |v| = |v|^2 rsq(|v|^2) and 1 / |v| from one transcendental (a quarter-rate
// instruction).
__device__ __forceinline__ float rsqf_hw(float x) { return __builtin_amdgcn_rsqf(x); }
// the larger value, or NaN if either is one (v_maximum3_f32)
__device__ __forceinline__ float max_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
// isGreater(a, b) with a, b >= 0 (util::isGreater, function.h, slack 1e-5 of
// the larger operand) reduces to a (1 - 1e-5) > b: one compare against a
// threshold scaled once per particle.
constexpr float REL_KEEP = 1.f - 1e-5f;

// entry t of a block
__device__ __forceinline__ int block_id(const uint4& b, int t) {
  const unsigned w = t < 2 ? b.x : t < 4 ? b.y : t < 6 ? b.z : b.w;
  return (int)((w >> ((t & 1) * 16)) & 0xffffu);
}

// Node data of the bond loops: the LDS window (LDS) or HBM.
//
// A neighbor is named by the 16-bit entry of the id list: the byte offset of
// its 16-byte LDS records (LDS tiles) or its id relative to the particle's
// first node (HBM tiles).
//
// LDS records, 16 bytes each, per window node:
//   lx  twice the FP32 position offset from the particle's first reference
//       node, and the volume over particle_scale
//                                       (first pass; with GEOM both passes)
//   lq  the displacement relative to the particle's first node in fixed
//       point (three int32 in units of a power-of-two step `us` chosen per
//       particle so that every value stays below 2^29 in magnitude), and the
//       node's alpha term (MixedArgs::fa)                     (first pass)
//   ly  the current position relative to that of the particle's first node,
//       in FP32 or, where that would cost accuracy, in fixed point (as lq,
//       with a step of its own), and the node's b term        (second pass)
// A bond's relative displacement is the exact integer difference of two lq
// records, rounded once to FP32 and scaled by us (exact): as accurate as
// rounding the FP64 difference to FP32, plus a quantisation of 2^-29 of the
// particle's largest relative displacement.  HBM tiles read the FP64 arrays
// (us = 1).
//
// The second pass takes only the direction of the current bond vector, the
// difference of two ly records.  While the particle is about as large as at
// the start (FIXED_FROM), FP32 positions are as accurate as the reference
// positions, which are FP32 throughout.  When its parts have flown apart
// they are not (sphere of 1021 nodes in two halves 1 m apart, strain 0.2: RMS
// force error 2.0e-5 of the largest force, 4.4e-6 in fixed point, which is the
// error of the displacement records), and the tile takes fixed point.  Fixed
// point throughout costs three conversions a bond: packing of 2000 spheres 3 %
// of the step, 512-instance ensemble 1.6 %.
//
// The record after the window's last node (offset 16 (we - ws)) stands for
// the list padding: a position so far off that its bond has no stretch, and
// weight 0, so the entries that fill up a lane's last block add nothing and
// the block loops need no test per bond.
constexpr float PAD_POS = 1.0e18f;
constexpr int PAD_Q = 1 << 30;  // its current position in fixed point (the nodes' are below 2^29)
// fixed point from this ratio of the largest component of the current
// positions to that of the reference positions on (a round body that turns
// stays at 1, a box reaches 1.7)
constexpr float FIXED_FROM = 1.25f;

template <int DIM, bool LDS>
struct Win {
  const char* lx;
  const char* lq;
  const char* ly;
  const DS* s;
  const MixedArgs* m;
  int gs;    // particle's first node
  int ws;    // window start
  float us;  // fixed-point step of the displacement records (1 for HBM tiles)
  double inv_scale;  // 1 / particle_scale
  double org[3];
  __device__ __forceinline__ int entry(int i) const { return LDS ? (i - ws) * 16 : i - gs; }
  __device__ __forceinline__ float4 x2(int e) const {
    if (LDS) return *(const float4*)(lx + e);
    const int64_t j = gs + e;
    return make_float4(2.f * (float)(s->xr[0][j] - org[0]), 2.f * (float)(s->xr[1][j] - org[1]),
                       DIM == 3 ? 2.f * (float)(s->xr[2][j] - org[2]) : 0.f, (float)(s->vol[j] * inv_scale));
  }
  // the node's own displacement record (fixed point) or displacement (FP64)
  struct Own {
    int q[3];
    double u[3];
    float a;
  };
  __device__ __forceinline__ Own own(int e) const {
    Own o{};
    if (LDS) {
      const int4 r = *(const int4*)(lq + e);
      o.q[0] = r.x;
      o.q[1] = r.y;
      o.q[2] = r.z;
      o.a = __int_as_float(r.w);
    } else {
      for (int d = 0; d < DIM; d++) o.u[d] = s->u[d][gs + e];
      o.a = m->fa[gs + e];
    }
    return o;
  }
  // relative displacement of neighbor e in units of us (FP32) and its alpha term
  __device__ __forceinline__ void du(int e, const Own& o, float* out, float& aj) const {
    if (LDS) {
      const int4 r = *(const int4*)(lq + e);
      out[0] = (float)(r.x - o.q[0]);
      out[1] = (float)(r.y - o.q[1]);
      if (DIM == 3) out[2] = (float)(r.z - o.q[2]);
      aj = __int_as_float(r.w);
    } else {
      for (int d = 0; d < DIM; d++) out[d] = (float)(s->u[d][gs + e] - o.u[d]);
      aj = m->fa[gs + e];
    }
  }
  // the node's own current position relative to the particle's first node
  // (FP32, fixed point or, HBM tiles, FP64) and its b term
  struct Cur {
    int4 r;
    double y[3];
  };
  __device__ __forceinline__ double pos(int64_t j, int d) const {
    return (s->xr[d][j] - org[d]) + (s->u[d][j] - s->u[d][gs]);
  }
  __device__ __forceinline__ Cur cur(int e) const {
    Cur o{};
    if (LDS) {
      o.r = *(const int4*)(ly + e);
    } else {
      for (int d = 0; d < DIM; d++) o.y[d] = pos(gs + e, d);
      o.r.w = __float_as_int(m->fb[gs + e]);
    }
    return o;
  }
  // current bond vector to neighbor e (in the unit of the records) and the
  // sum of the b terms
  template <bool FIXED>
  __device__ __forceinline__ void dy(int e, const Cur& o, float* out, float& b) const {
    float bj;
    if (LDS) {
      const int4 r = *(const int4*)(ly + e);
      auto diff = [](int x, int y) { return FIXED ? (float)(x - y) : __int_as_float(x) - __int_as_float(y); };
      out[0] = diff(r.x, o.r.x);
      out[1] = diff(r.y, o.r.y);
      if (DIM == 3) out[2] = diff(r.z, o.r.z);
      bj = __int_as_float(r.w);
    } else {
      for (int d = 0; d < DIM; d++) out[d] = (float)(pos(gs + e, d) - o.y[d]);
      bj = m->fb[gs + e];
    }
    b = __int_as_float(o.r.w) + bj;
  }
};

__device__ __forceinline__ float round_up(double a) { return (float)(a * (1.0 + 0x1p-20)); }
// Largest components over a particle's nodes, relative to its first node: the
// displacement and the current position
struct PartMax {
  double u = 0., y = 0.;
  template <int DIM>
  __device__ __forceinline__ void node(const double* xd, const double* du) {
    for (int d = 0; d < DIM; d++) {
      u = fmax(u, fabs(du[d]));
      y = fmax(y, fabs(xd[d] + du[d]));
    }
  }
  // the workgroup's maxima as floats rounded up (the fixed-point steps only
  // have to bound them); they do not depend on the order, so every tile of a
  // particle gets the same values
  __device__ __forceinline__ float2 group(float2* red) const {
    float2 m = make_float2(round_up(u), round_up(y));
    auto join = [&](float a, float b) { m = make_float2(fmaxf(m.x, a), fmaxf(m.y, b)); };
    for (int o = WAVE / 2; o > 0; o >>= 1) join(__shfl_xor(m.x, o), __shfl_xor(m.y, o));
    if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = m;
    __syncthreads();
    for (int w = 0; w < (int)(blockDim.x / WAVE); w++) join(red[w].x, red[w].y);
    return m;
  }
};

// the maxima of the particles with open LDS tiles: one workgroup each
template <int DIM>
__global__ void __launch_bounds__(1024) k_mixed_umax(DS s, MixedArgs m) {
  __shared__ float2 red[1024 / WAVE];
  const int pid = m.open_pids[blockIdx.x];
  const DevParticle& p = s.P[pid];
  const int64_t gs = p.glob_start;
  PartMax mx;
  for (int64_t j = gs + threadIdx.x; j < p.glob_end; j += blockDim.x) {
    double xd[3], du[3];
    for (int d = 0; d < DIM; d++) {
      xd[d] = s.xr[d][j] - s.xr[d][gs];
      du[d] = s.u[d][j] - s.u[d][gs];
    }
    mx.node<DIM>(xd, du);
  }
  const float2 mf = mx.group(red);
  if (threadIdx.x == 0) m.pmax[pid] = mf;
}

// the smallest power of two 2^e with mf / 2^e < 2^29 (e >= -126: a window at
// rest keeps all zeros)
__device__ __forceinline__ int fixed_exp(float mf) {
  if (!(mf > 0.f)) return -126;
  int ex;
  frexpf(mf, &ex);  // mf < 2^ex
  return ex - 29 > -126 ? ex - 29 : -126;
}

// Stage a tile's window in LDS: the records that the pass (or, FIRST and
// SECOND, both passes) reads.  The fixed-point steps come from the largest
// values of the whole particle, so that the records, and the results, do not
// depend on the tile shape; a closed tile (the whole particle) takes them over
// its window, an open tile reads them from k_mixed_umax.  The b terms of the
// fused kernel are written by its first pass; those of an open tile come from
// the other kernel.
// Returns the displacements' step us; fixed: ly is in fixed point.
template <int DIM, bool FIRST, bool SECOND, bool GEOM>
__device__ __forceinline__ float stage_window(const DS& s, const MixedArgs& m, const DevTile& t, float4* lx,
                                              int4* lq, int4* ly, const double* org, double inv_scale,
                                              float2* red, bool& fixed) {
  const int nw = t.we - t.ws;
  const int gs = (int)s.P[t.pid].glob_start;
  double u0[3] = {0., 0., 0.};
  for (int d = 0; d < DIM; d++) u0[d] = s.u[d][gs];
  constexpr bool CLOSED = FIRST && SECOND;
  float2 mf = make_float2(0.f, 0.f);
  if (!CLOSED) mf = m.pmax[t.pid];
  PartMax mx;
  for (int q = threadIdx.x; q < nw; q += blockDim.x) {
    const int j = t.ws + q;
    double xd[3] = {0., 0., 0.}, du[3] = {0., 0., 0.};
    for (int d = 0; d < DIM; d++) xd[d] = s.xr[d][j] - org[d];
    if (FIRST || GEOM)
      lx[q] = make_float4(2.f * (float)xd[0], 2.f * (float)xd[1], 2.f * (float)xd[2], (float)(s.vol[j] * inv_scale));
    if (SECOND) {
      for (int d = 0; d < DIM; d++) du[d] = s.u[d][j] - u0[d];
      if (CLOSED) mx.node<DIM>(xd, du);
      ly[q] = make_int4(__float_as_int((float)(xd[0] + du[0])), __float_as_int((float)(xd[1] + du[1])),
                        __float_as_int((float)(xd[2] + du[2])), FIRST ? 0 : __float_as_int(m.fb[j]));
    }
  }
  if (CLOSED) mf = mx.group(red);
  fixed = __builtin_amdgcn_readfirstlane(mf.y > FIXED_FROM * m.part[t.pid].xmax);
  const int eu = fixed_exp(mf.x);
  if (FIRST) {
    const double inv_us = ldexp(1., -eu);
    for (int q = threadIdx.x; q < nw; q += blockDim.x) {
      const int j = t.ws + q;
      int qq[3] = {0, 0, 0};
      for (int d = 0; d < DIM; d++) qq[d] = (int)rint((s.u[d][j] - u0[d]) * inv_us);
      lq[q] = make_int4(qq[0], qq[1], qq[2], __float_as_int(m.fa[j]));
    }
  }
  if (SECOND && fixed) {
    const double inv_ys = ldexp(1., -fixed_exp(mf.y));
    for (int q = threadIdx.x; q < nw; q += blockDim.x) {
      const int j = t.ws + q;
      int yy[3] = {0, 0, 0};
      for (int d = 0; d < DIM; d++) yy[d] = (int)rint(((s.xr[d][j] - org[d]) + (s.u[d][j] - u0[d])) * inv_ys);
      ly[q] = make_int4(yy[0], yy[1], yy[2], ly[q].w);
    }
  }
  if (threadIdx.x == 0) {  // the padding's record
    const int pad = fixed ? PAD_Q : __float_as_int(PAD_POS);
    if (FIRST || GEOM) lx[nw] = make_float4(PAD_POS, PAD_POS, DIM == 3 ? PAD_POS : 0.f, 0.f);
    if (FIRST) lq[nw] = make_int4(0, 0, 0, 0);
    if (SECOND) ly[nw] = make_int4(pad, pad, DIM == 3 ? pad : 0, 0);
  }
  __syncthreads();
  return ldexpf(1.f, eu);
}

// Per-particle constants of the mixed bond loops (those of every bond in
// scalar registers)
struct StateConsts {
  float thr4;      // |S| / 4 > thr4: the bond breaks (isGreater(|S|, s0 + 1e-10))
  float inv_s0, Kn, Rc;
  double K, G, scale;
  // GEOM: J = ja + jb r2 (constant and linear influence functions), volume
  // correction up_h - r2 inv_h2 where r2 > low2
  float ja, jb, low2, inv_h2, up_h;
  __device__ StateConsts(const DS& s, const MixedArgs& m, int pid) {
    const DevParticle& p = s.P[pid];
    thr4 = uniform(0.25f * ((float)(p.mat[2] + 1.0e-10) / REL_KEEP));
    inv_s0 = uniform((float)(1.0 / p.mat[2]));
    Rc = uniform((float)p.Rc);
    K = p.mat[0];
    G = p.mat[1];
    scale = m.part[pid].scale;
    Kn = uniform((float)(p.Kn * scale));
    ja = uniform((float)s.inf_p0);
    jb = uniform(s.inf_type == 1 ? (float)(0.5 * s.inf_p1 / p.horizon) : 0.f);
    low2 = uniform(2.f * ((float)(p.horizon - 0.5 * p.h) / REL_KEEP));
    inv_h2 = uniform((float)(0.5 / p.h));
    up_h = uniform((float)((p.horizon + 0.5 * p.h) / p.h));
  }
  // GEOM: the weight 2 r J V^c / scale of a bond of length r2 / 2 whose
  // neighbor has volume v scale.  The padding's length (Win) makes J a large
  // number, but a finite one in any unit of length: the scale, which goes with
  // the fourth power of the mesh size, is in v, which is 0 there.  The
  // correction is 1 at the distance horizon - h/2 from which it applies, so
  // clamping it to [0, 1], which the multiply-add does for nothing, saves the
  // compare and the select (exact) for every bond but those in the slack of
  // the reference's compare (see slack_bond).
  __device__ __forceinline__ float weight(float r2, float v, bool exact) const {
#pragma clang fp contract(fast)
    const float c = up_h - r2 * inv_h2;
    float k = __builtin_amdgcn_fmed3f(c, 0.f, 1.f);
    if (exact) k = r2 > low2 ? c : 1.f;
    return r2 * ((ja + jb * r2) * (v * k));
  }
};

// A bond whose length r is above low = horizon - h/2 by less than the slack
// 1e-5 r of the reference's compare keeps its full volume, where the formula
// gives up to 1e-5 low / h less.  Its 8-bond block is marked in the LDS tiles'
// lists (SLACK_BLOCK in the block's first entry, whose value stays below it)
// and takes the exact form.  (Within 2^-24 of low the two agree to rounding;
// the upper end is taken with a margin.)
constexpr unsigned SLACK_BLOCK = 0x8000u;
__device__ __forceinline__ bool slack_bond(double r, double low) {
  return r > low * (1. + 0x1p-24) && r < low * (1. + 1.2 * COMPARE_EPS);
}

// The two passes of a node (dilation, demModel.cpp:610-679; force, :682-788
// with PdState::getBondEF, material.h:1415-1429) in mixed precision.
//
// With ef_i + ef_j = J (r (b_i + b_j) + c (alpha_i + alpha_j)), c = |y| - |xi|
// the change of length, y = xi + eta and b = theta (3K/m - alpha / 3), only
// the b terms of the force need the dilation of the neighbors; alpha is
// constant.  So the first pass, which has the accurate change of length
//   c = (2 xi.eta + eta.eta) / (|y| + |xi|)
// at hand, also sums the alpha part of the force and the repulsion of broken
// bonds (into f), and the second pass only adds
//   sum_j r J V_j^c (b_i + b_j) y / |y|
// from the bond's weight and the neighbors' current positions.
//
// The loops are bound by FP32 instruction issue and the latency of the list
// reads.  Per bond in 3D they take 42 VALU instructions in the first pass and 14
// in the second with weights from the lists, 47 and 28 evaluating them (of which
// 3 and 1 or 2 are half-rate transcendentals); with the reference geometry
// evaluated in both passes and the alpha part in the second they took 57 each.
// Packing of 2000 spheres (weights evaluated), both passes of a step: 409 us with
// the alpha part in the second, 328 us now (kernel trace), 412 MB against 134 MB
// fetched.
//
// The loops take 4 bonds at a time without any test per bond: the lists are
// padded to whole blocks (see Win), and a block whose largest stretch says that
// a bond breaks now is done again with tests.  Where a lane of the wavefront
// holds a broken bond among the 32 of a word, all its lanes take those blocks
// with tests only, two bonds a round: doing the blocks twice there, lane by
// lane and bond by bond, took 211 us for both passes of 400 spheres of 1021
// nodes with 5 % of their bonds broken, 126 us now (104 us with none broken);
// 2000 disks of 361 nodes 132 us, 89 now (77).  (A fully unrolled loop with
// tests takes 120 us there, but its registers spill in the loop without tests:
// 8 % on the intact packing of 2000 spheres, 26 % on the 512-instance ensemble.
// The looking for broken bits costs 1 % of these steps.)
// Every sum is taken per block (theta in FP64, forces in FP32) and the blocks
// are added in list order in FP64, so the results do not depend on how blocks
// are dealt to lanes.

// one bond of the first pass: doubled lengths, the quarter stretch and the
// doubled current bond vector
template <int DIM>
struct Stretch {
  float xx4, yy4, r2, inv_r2, l2, inv_l2, c2, y2[3];
  // d2: twice the reference bond vector; q: relative displacement in units of us
  __device__ __forceinline__ Stretch(const float* d2, const float* q, float us) {
#pragma clang fp contract(fast)
    float t = q[0] * (d2[0] + us * q[0]);
    xx4 = d2[0] * d2[0];
    for (int d = 1; d < DIM; d++) {
      xx4 += d2[d] * d2[d];
      t += q[d] * (d2[d] + us * q[d]);
    }
    for (int d = 0; d < DIM; d++) y2[d] = d2[d] + 2.f * us * q[d];
    t *= us;                      // |y|^2 - |xi|^2
    yy4 = xx4 + 4.f * t;
    inv_r2 = rsqf_hw(xx4);
    inv_l2 = rsqf_hw(yy4);
    r2 = xx4 * inv_r2;            // 2 |xi|
    l2 = yy4 * inv_l2;            // 2 |y|
    c2 = t * rcpf(l2 + r2);       // (|y| - |xi|) / 2
  }
  // a bond whose ends have met (|y| = 0 to rounding: l2 above is no number) has
  // lost its whole length
  __device__ __forceinline__ void met() {
    if (yy4 <= 0.f) {
      l2 = 0.f;
      c2 = -0.25f * r2;
    }
  }
};

// the sums of one 8-bond block in the first pass
struct Block1 {
  double theta;  // sum r c J V^c / particle_scale
  float f[3];
  float z;       // largest |S| / 4, NaN if one is
};

// First pass of one block of a node's list: entries `cur`, weights at wg,
// `left` bonds to the list's end, broken bits wblk; brk gets the bonds that
// break now.  `tests` (the same for the wavefront): some lane has a broken bond
// here or hereabouts, and the block goes to the loop with tests at once.
template <int DIM, bool LDS, bool GEOM>
__device__ __forceinline__ Block1 first_block(const Win<DIM, LDS>& w, const StateConsts& c, uint4 cur,
                                              const float4* wg, int left, unsigned wblk, const float* xi,
                                              const typename Win<DIM, LDS>::Own& own, float us, bool tests, unsigned& brk) {
#pragma clang fp contract(fast)
  Block1 o{0., {0.f, 0.f, 0.f}, 0.f};
  const bool slack = GEOM && (!LDS || (cur.x & SLACK_BLOCK));
  // one bond; SURE that it is whole and stays so
  auto bond = [&](const int e, const float wt, const int tt, auto sure) {
    constexpr bool SURE = decltype(sure)::value;
    const float4 xvj = w.x2(e);
    const float xj[3] = {xvj.x, xvj.y, xvj.z};
    float d2[3], du[3], aj;
    w.du(e, own, du, aj);
    for (int d = 0; d < DIM; d++) d2[d] = xj[d] - xi[d];
    Stretch<DIM> b(d2, du, us);
    if (!SURE) b.met();
    const float wj = GEOM ? c.weight(b.r2, xvj.w, !SURE && slack) : wt;
    const float p = b.c2 * b.inv_r2;  // S / 4
    o.z = max_nan(o.z, fabsf(p));
    const float th = b.c2 * wj;
    float sf = p * wj * (own.a + aj) * b.inv_l2;
    if (SURE) {
      o.theta += (double)th;
    } else {
      bool fs = ((wblk >> tt) & 1u) != 0u;
      if (!fs && fabsf(p) > c.thr4) {
        fs = true;
        brk |= 1u << tt;
      }
      if (!fs) {
        o.theta += (double)th;
      } else {
        // Kn V (|y| - Rc) y / |y| where it repels (Kn with the scale of vj)
        sf = c.Kn * xvj.w * (0.5f * b.l2 - c.Rc) * b.inv_l2;
        if (sf > 0.f) sf = 0.f;
      }
    }
    for (int d = 0; d < DIM; d++) o.f[d] += sf * b.y2[d];
  };
  if (LDS && !tests) {
    auto half = [&](unsigned id0, unsigned id1, const float4& wt, const int t0) {
      const std::true_type sure{};
      bond((int)(id0 & 0x7fffu), wt.x, t0, sure);
      bond((int)(id0 >> 16), wt.y, t0 + 1, sure);
      pin(o.f, o.z);
      bond((int)(id1 & 0xffffu), wt.z, t0 + 2, sure);
      bond((int)(id1 >> 16), wt.w, t0 + 3, sure);
      pin(o.f, o.z);
    };
    const float4 none = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 wa = GEOM ? none : wg[0], wb = GEOM ? none : wg[WAVE];
    half(cur.x, cur.y, wa, 0);
    if (left > KB / 2) half(cur.z, cur.w, wb, KB / 2);
    if (o.z <= c.thr4 && !slack) return o;
    o = Block1{0., {0.f, 0.f, 0.f}, 0.f};
  }
  if (!LDS) {
#pragma unroll
    for (int tt = 0; tt < KB; tt++)
      if (tt < left) bond(block_id(cur, tt), GEOM ? 0.f : ((const float*)(wg + (tt / 4) * WAVE))[tt % 4], tt, std::false_type{});
    return o;
  }
  // with tests, two entries at a time: blocks with a bond that breaks now or
  // has no length left or (GEOM) is in the slack, and those of a wavefront that
  // holds broken bonds
#pragma unroll 1
  for (int tt = 0; tt < KB && tt < left; tt += 2) {
    float2 wt = make_float2(0.f, 0.f);
    if (!GEOM) wt = *(const float2*)((const float*)(wg + (tt / 4) * WAVE) + tt % 4);
    bond((int)(cur.x & 0x7fffu), wt.x, tt, std::false_type{});
    pin(o.f, o.z);
    bond((int)(cur.x >> 16), wt.y, tt + 1, std::false_type{});
    cur.x = cur.y;
    cur.y = cur.z;
    cur.z = cur.w;
  }
  return o;
}

// A node's list may be dealt to LPN neighboring lanes (LPN 1, 4 or 8: a
// 32-bit bond word's four blocks are then taken at once): lane `sub` takes
// blocks sub, sub + LPN, ...; the group's lanes then all add the blocks' sums
// in list order, so every lane holds the node's sums.  (value of group lane k)
template <int LPN, class T>
__device__ __forceinline__ T group_lane(T v, int k) {
  return LPN == 1 ? v : __shfl(v, k, LPN);
}

// First pass of the node in thread slot q: breaks bonds, writes theta, the
// damage Z and the first part of the force, and returns the node's b term.
// The damage Z_i (demModel.cpp:770-773) is the plain maximum of |S| / s0 over
// the list, broken bonds included, NaN where a stretch is (the reference's running compare with a
// 1e-5 relative slack keeps a value at most 1e-5 below it; FP32 bond
// arithmetic is the larger difference).
template <int DIM, bool LDS, bool GEOM, int LPN>
__device__ __forceinline__ float first_pass_node(const DS& s, const MixedArgs& m, const DevTile& t,
                                                 const Win<DIM, LDS>& w, const StateConsts& c, int q, int& node) {
  const uint32_t ln = m.lnode[t.node + q];
  const int i = t.ts + (int)(ln & 0xffffu), n = (int)(ln >> 16);
  node = i;
  const int sub = LPN == 1 ? 0 : (int)(threadIdx.x % LPN);
  const int ei = w.entry(i);
  const int64_t at = t.data + m.lslice[t.slice + q / WAVE];
  const uint4* cb = (const uint4*)(m.col16 + at) + q % WAVE;
  const float4* wb = (const float4*)(m.wgt + at) + q % WAVE;
  unsigned* bw = s.bits + s.bptr[i / WAVE] + i % WAVE;
  const float4 xvi = w.x2(ei);
  const float xi[3] = {xvi.x, xvi.y, xvi.z};
  const auto own = w.own(ei);
  const float us = uniform(w.us);
  double theta = 0., force[3] = {0., 0., 0.};
  float Zs = 0.f;  // maximum of |S| / 4 over all bonds, broken ones included
  auto add = [&](const Block1& o, int k) {
    theta += group_lane<LPN>(o.theta, k);
    Zs = max_nan(Zs, group_lane<LPN>(o.z, k));
    for (int d = 0; d < DIM; d++) force[d] += (double)group_lane<LPN>(o.f[d], k);
  };
  if (LPN == 1) {
    unsigned word = 0, wnew = 0;
    bool tests = false;  // a lane of the wavefront holds a broken bond among these 32
    uint4 blk = n > 0 ? cb[0] : make_uint4(0, 0, 0, 0);
    for (int kb = 0; kb < n; kb += KB) {
      if ((kb & 31) == 0) {
        if (kb > 0 && wnew != word) bw[(int64_t)((kb >> 5) - 1) * WAVE] = wnew;
        word = bw[(int64_t)(kb >> 5) * WAVE];
        wnew = word;
        tests = __any(word != 0u);
      }
      const uint4 cur = blk;
      if (kb + KB < n) blk = cb[(kb / KB + 1) * WAVE];
      unsigned brk = 0;
      const Block1 o = first_block<DIM, LDS, GEOM>(w, c, cur, wb + (kb / KB) * 2 * WAVE, n - kb,
                                             (word >> (kb & 31)) & 0xffu, xi, own, us, tests, brk);
      wnew |= brk << (kb & 31);
      add(o, 0);
    }
    if (n > 0 && wnew != word) bw[(int64_t)((n - 1) >> 5) * WAVE] = wnew;
  } else {
    for (int k0 = 0; k0 < n; k0 += KB * LPN) {
      const int kb = k0 + KB * sub;
      Block1 o{0., {0.f, 0.f, 0.f}, 0.f};
      unsigned word = 0, brk = 0;
      if (kb < n) {
        word = bw[(int64_t)(kb >> 5) * WAVE];
        o = first_block<DIM, LDS, GEOM>(w, c, cb[(kb / KB) * WAVE], wb + (kb / KB) * 2 * WAVE, n - kb,
                                  (word >> (kb & 31)) & 0xffu, xi, own, us, true, brk);
      }
      for (int k = 0; k < LPN; k++)
        if (k0 + KB * k < n) add(o, k);
      // the breaks of a word's four blocks joined, written by their first lane
      unsigned b = brk << (kb & 31);
      b |= (unsigned)__shfl_xor((int)b, 1, LPN);
      b |= (unsigned)__shfl_xor((int)b, 2, LPN);
      if (kb < n && b != 0u && (sub & 3) == 0) bw[(int64_t)(kb >> 5) * WAVE] = word | b;
    }
  }
  const double mi = s.mx[i];
  const double th = 3. * (c.scale * theta) / mi;
  if (sub == 0) {
    s.theta[i] = th;
    s.Z[i] = 4.f * Zs * c.inv_s0;
    for (int d = 0; d < DIM; d++) s.f[d][i] = force[d];
  }
  const double alpha = 15. * c.G / mi;
  return (float)(c.scale * (th * ((3. * c.K / mi) - alpha / 3.)));
}

// Second pass of one block: sum of 2 r J V^c (b_i + b_j) y / |y| into f
template <int DIM, bool LDS, bool GEOM, bool FIXED>
__device__ __forceinline__ void second_block(const Win<DIM, LDS>& w, const StateConsts& c, const uint4& cur,
                                             const float4* wg, int left, unsigned wblk, const float* xi,
                                             const typename Win<DIM, LDS>::Cur& own, bool tests, float (&f)[3]) {
#pragma clang fp contract(fast)
  // one bond (whole: SURE that it is not broken)
  auto bond = [&](const int tt, const float wt, auto whole, auto exact) {
    const int e = block_id(cur, tt) & (LDS ? 0x7fff : 0xffff);  // (the first entry's top bit in LDS tiles: SLACK_BLOCK)
    float wj = wt;
    if (GEOM) {
      const float4 xvj = w.x2(e);
      const float xj[3] = {xvj.x, xvj.y, xvj.z};
      float d2 = xj[0] - xi[0], xx4 = d2 * d2;
      for (int d = 1; d < DIM; d++) {
        d2 = xj[d] - xi[d];
        xx4 += d2 * d2;
      }
      wj = c.weight(xx4 * rsqf_hw(xx4), xvj.w, decltype(exact)::value);
    }
    float y[3], b;
    w.template dy<FIXED>(e, own, y, b);
    float yy = y[0] * y[0];
    for (int d = 1; d < DIM; d++) yy += y[d] * y[d];
    float sf = wj * b * rsqf_hw(yy);
    if (!decltype(whole)::value) sf = ((wblk >> tt) & 1u) ? 0.f : sf;  // (broken bonds: in the first pass)
    for (int d = 0; d < DIM; d++) f[d] += sf * y[d];
  };
  const std::true_type yes{};
  const std::false_type no{};
  if (LDS && !(GEOM && (cur.x & SLACK_BLOCK))) {
    const float4 wa = GEOM ? make_float4(0.f, 0.f, 0.f, 0.f) : wg[0];
    const float4 wb = GEOM ? make_float4(0.f, 0.f, 0.f, 0.f) : wg[WAVE];
    auto half = [&](int t0, const float4& wt, auto whole) {
      bond(t0, wt.x, whole, no);
      bond(t0 + 1, wt.y, whole, no);
      if (GEOM) pin(f, f[0]);
      bond(t0 + 2, wt.z, whole, no);
      bond(t0 + 3, wt.w, whole, no);
    };
    auto block = [&](auto whole) {
      half(0, wa, whole);
      pin(f, f[0]);
      if (left > KB / 2) half(KB / 2, wb, whole);
    };
    if (!tests)
      block(yes);
    else if (wblk != (left < KB ? (1u << left) - 1u : 0xffu))  // (not all of them broken)
      block(no);
    return;
  }
  if (!LDS) {
#pragma unroll
    for (int tt = 0; tt < KB; tt++)
      if (tt < left && !((wblk >> tt) & 1u))
        bond(tt, GEOM ? 0.f : ((const float*)(wg + (tt / 4) * WAVE))[tt % 4], yes, yes);
    return;
  }
#pragma unroll 1
  for (int tt = 0; tt < KB && tt < left; tt++) bond(tt, 0.f, no, yes);  // (GEOM, in the slack)
}

// Second pass of the node in thread slot q: adds the b terms to f.
template <int DIM, bool LDS, bool GEOM, bool FIXED, int LPN>
__device__ __forceinline__ void second_pass_node(const DS& s, const MixedArgs& m, const DevTile& t,
                                                 const Win<DIM, LDS>& w, const StateConsts& c, int q) {
  const uint32_t ln = m.lnode[t.node + q];
  const int i = t.ts + (int)(ln & 0xffffu), n = (int)(ln >> 16);
  const int sub = LPN == 1 ? 0 : (int)(threadIdx.x % LPN);
  const int64_t at = t.data + m.lslice[t.slice + q / WAVE];
  const uint4* cb = (const uint4*)(m.col16 + at) + q % WAVE;
  const float4* wb = (const float4*)(m.wgt + at) + q % WAVE;
  const unsigned* bw = s.bits + s.bptr[i / WAVE] + i % WAVE;
  const auto own = w.cur(w.entry(i));
  const float4 xvi = GEOM ? w.x2(w.entry(i)) : make_float4(0.f, 0.f, 0.f, 0.f);
  const float xi[3] = {xvi.x, xvi.y, xvi.z};
  double force[3] = {0., 0., 0.};
  for (int d = 0; d < DIM; d++) force[d] = s.f[d][i];
  if (LPN == 1) {
    unsigned word = 0;
    bool tests = false;
    uint4 blk = n > 0 ? cb[0] : make_uint4(0, 0, 0, 0);
    for (int kb = 0; kb < n; kb += KB) {
      if ((kb & 31) == 0) {
        word = bw[(int64_t)(kb >> 5) * WAVE];
        tests = __any(word != 0u);
      }
      const uint4 cur = blk;
      if (kb + KB < n) blk = cb[(kb / KB + 1) * WAVE];
      float fb[3] = {0.f, 0.f, 0.f};
      second_block<DIM, LDS, GEOM, FIXED>(w, c, cur, wb + (kb / KB) * 2 * WAVE, n - kb, (word >> (kb & 31)) & 0xffu, xi, own,
                                   tests, fb);
      for (int d = 0; d < DIM; d++) force[d] += 0.5 * (double)fb[d];
    }
  } else {
    for (int k0 = 0; k0 < n; k0 += KB * LPN) {
      const int kb = k0 + KB * sub;
      float fb[3] = {0.f, 0.f, 0.f};
      if (kb < n)
        second_block<DIM, LDS, GEOM, FIXED>(w, c, cb[(kb / KB) * WAVE], wb + (kb / KB) * 2 * WAVE, n - kb,
                                     (bw[(int64_t)(kb >> 5) * WAVE] >> (kb & 31)) & 0xffu, xi, own, true, fb);
      for (int k = 0; k < LPN; k++)
        if (k0 + KB * k < n)
          for (int d = 0; d < DIM; d++) force[d] += 0.5 * (double)group_lane<LPN>(fb[d], k);
    }
  }
  if (sub == 0)
    for (int d = 0; d < DIM; d++) s.f[d][i] = force[d];
}

// Tile ranges of MixedArgs::tiles: closed LDS tiles (whole particles, fused
// kernel), open LDS tiles, HBM tiles.  An HBM tile is shared by hbm_split
// workgroups of HBM_TPB threads (there is no window to stage).  Workgroups go
// to the 8 XCDs in turn; an XCD takes an eighth of the tiles, one after the
// other with all of their workgroups (the last may find fewer: hbm_blocks()
// workgroups, hbm_tile() beyond the tiles).
constexpr int XCDS = 8;
__host__ __device__ inline int hbm_per_xcd(const MixedArgs& m) { return (m.ntiles_hbm + XCDS - 1) / XCDS; }
__host__ inline unsigned hbm_blocks(const MixedArgs& m) { return (unsigned)(XCDS * hbm_per_xcd(m) * m.hbm_split); }
__device__ __forceinline__ int hbm_tile(const MixedArgs& m) {
  return (int)blockIdx.x % XCDS * hbm_per_xcd(m) + (int)blockIdx.x / XCDS / m.hbm_split;
}
template <bool LDS>
__device__ __forceinline__ const DevTile& tile_of(const MixedArgs& m) {
  return m.tiles[m.ntiles_closed + (LDS ? (int)blockIdx.x : m.ntiles_lds + hbm_tile(m))];
}
// thread slot of the workgroup's round `it` over the tile's slots (LPN lanes per slot)
template <bool LDS, int LPN>
__device__ __forceinline__ int slot_of(const MixedArgs& m, int it) {
  const int part = LDS ? 0 : (int)blockIdx.x / XCDS % m.hbm_split;
  return ((LDS ? it : it * m.hbm_split + part) * (int)blockDim.x + (int)threadIdx.x) / LPN;
}
template <bool LDS, int LPN>
__device__ __forceinline__ int slot_rounds(const MixedArgs& m, const DevTile& t) {
  const int per = (int)blockDim.x / LPN * (LDS ? 1 : m.hbm_split);
  return (t.te - t.ts + per - 1) / per;
}

// the second pass of a tile's nodes
template <int DIM, bool LDS, bool GEOM, int LPN>
__device__ __forceinline__ void second_pass(const DS& s, const MixedArgs& m, const DevTile& t, const Win<DIM, LDS>& w,
                                            const StateConsts& c, bool fixed) {
  const int nr = slot_rounds<LDS, LPN>(m, t);
  auto run = [&](auto fx) {
    for (int it = 0; it < nr; it++) {
      const int q = slot_of<LDS, LPN>(m, it);
      if (q < t.te - t.ts) second_pass_node<DIM, LDS, GEOM, decltype(fx)::value, LPN>(s, m, t, w, c, q);
    }
  };
  if (LDS && fixed)
    run(std::true_type{});
  else
    run(std::false_type{});
}

// LDS of the window records, one more than the window for the list padding
// (LDS tiles), or a dummy (HBM tiles)
#define PDEM_WINDOW_LDS(LDS_ON, NODES, FIRST, SECOND, GEOM)    \
  __shared__ float4 lx[(LDS_ON) && ((FIRST) || (GEOM)) ? (NODES) + 1 : 1]; \
  __shared__ int4 lq[(LDS_ON) && (FIRST) ? (NODES) + 1 : 1];   \
  __shared__ int4 ly[(LDS_ON) && (SECOND) ? (NODES) + 1 : 1];  \
  __shared__ float2 red[1024 / WAVE];
#define PDEM_WINDOW(DIM, LDS_ON, t, gs) \
  Win<DIM, LDS_ON> w{(const char*)lx, (const char*)lq, (const char*)ly, &s, &m, gs, t.ws, 1.f, \
                      m.part[t.pid].inv_scale, {0., 0., 0.}}; \
  for (int d = 0; d < DIM; d++) w.org[d] = s.xr[d][gs];

// First pass of the open tiles (tiles that do not hold a whole particle:
// the second pass of a tile reads the b terms of nodes of other tiles).
template <int DIM, bool LDS, bool GEOM, int TPB, int NODES = LDS_NODES, int LPN = 1>
__global__ void __launch_bounds__(TPB, LDS ? MIXED_WAVES_PER_SIMD : HBM_WAVES_PER_SIMD) k_mixed_dilation(DS s, MixedArgs m) {
  if (!LDS && hbm_tile(m) >= m.ntiles_hbm) return;
  PDEM_WINDOW_LDS(LDS, NODES, true, false, GEOM)
  const DevTile t = tile_of<LDS>(m);
  const DevParticle& p = s.P[t.pid];
  const int gs = (int)p.glob_start;
  PDEM_WINDOW(DIM, LDS, t, gs)
  bool fixed = false;
  if (LDS) w.us = stage_window<DIM, true, false, GEOM>(s, m, t, lx, lq, ly, w.org, w.inv_scale, red, fixed);
  const StateConsts c(s, m, t.pid);
  const int nr = slot_rounds<LDS, LPN>(m, t);
  for (int it = 0; it < nr; it++) {
    const int q = slot_of<LDS, LPN>(m, it);
    if (q >= t.te - t.ts) continue;
    int i;
    const float b = first_pass_node<DIM, LDS, GEOM, LPN>(s, m, t, w, c, q, i);
    if (LPN == 1 || threadIdx.x % LPN == 0) m.fb[i] = b;
  }
}

// Second pass of the open tiles.
template <int DIM, bool LDS, bool GEOM, int TPB, int NODES = LDS_NODES, int LPN = 1>
__global__ void __launch_bounds__(TPB, LDS ? MIXED_WAVES_PER_SIMD : HBM_WAVES2_PER_SIMD) k_mixed_force(DS s, MixedArgs m) {
  if (!LDS && hbm_tile(m) >= m.ntiles_hbm) return;
  PDEM_WINDOW_LDS(LDS, NODES, false, true, GEOM)
  const DevTile t = tile_of<LDS>(m);
  const DevParticle& p = s.P[t.pid];
  const int gs = (int)p.glob_start;
  PDEM_WINDOW(DIM, LDS, t, gs)
  bool fixed = false;
  if (LDS) stage_window<DIM, false, true, GEOM>(s, m, t, lx, lq, ly, w.org, w.inv_scale, red, fixed);
  const StateConsts c(s, m, t.pid);
  second_pass<DIM, LDS, GEOM, LPN>(s, m, t, w, c, fixed);
}

// Both passes of a closed tile, a whole particle, so that every neighbor of
// its nodes is one of its nodes, in one workgroup: the window is staged in
// LDS once, the first pass leaves each node's b term in its LDS record, and
// after a barrier the second pass reads them there.
template <int DIM, bool GEOM, int TPB, int NODES = LDS_NODES>
__global__ void __launch_bounds__(TPB, TPB == 512 ? 6 : MIXED_WAVES_PER_SIMD) k_mixed_state(DS s, MixedArgs m) {
  PDEM_WINDOW_LDS(true, NODES, true, true, GEOM)
  const DevTile t = m.tiles[blockIdx.x];
  const DevParticle& p = s.P[t.pid];
  const int gs = (int)p.glob_start;
  PDEM_WINDOW(DIM, true, t, gs)
  bool fixed;
  w.us = stage_window<DIM, true, true, GEOM>(s, m, t, lx, lq, ly, w.org, w.inv_scale, red, fixed);
  const StateConsts c(s, m, t.pid);
  const int nr = slot_rounds<true, 1>(m, t);
  for (int it = 0; it < nr; it++) {
    const int q = slot_of<true, 1>(m, it);
    if (q >= t.te - t.ts) continue;
    int i;
    const float b = first_pass_node<DIM, true, GEOM, 1>(s, m, t, w, c, q, i);
    ly[i - t.ws].w = __float_as_int(b);
  }
  __syncthreads();
  second_pass<DIM, true, GEOM, 1>(s, m, t, w, c, fixed);
}

#undef PDEM_WINDOW
#undef PDEM_WINDOW_LDS

// the force reset of nodes that take no PD force (a list built at set-up);
// grid-stride
constexpr int BZ_BLOCKS = 1024;
template <int DIM>
__global__ void k_zero_noforce(DS s) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = gid(); k < s.n_noforce; k += stride) {
    const int64_t i = s.noforce_nodes[k];
    for (int d = 0; d < DIM; d++) s.f[d][i] = 0.;
  }
}

// Set-up of the lists (see DevTile).

// whether a tile's list has weights: where it reads them (HBM tiles evaluate
// theirs but for the Gaussian influence function's)
__device__ __forceinline__ bool has_weights(const DS& s, const MixedArgs& m, const DevTile& t) {
  return s.inf_type == 2 || (t.lds && !m.geom);
}

// weight 2 r J(r) V_j^c / particle_scale of a bond (materialUtil.cpp:21-73, m_x's terms)
template <int DIM>
__device__ __forceinline__ double bond_weight(const DS& s, const DevParticle& p, double inv_scale, int i, int j,
                                              bool& slack) {
  double dx[3];
  for (int d = 0; d < DIM; d++) dx[d] = s.xr[d][j] - s.xr[d][i];
  const double r = len3<DIM>(dx);
  double v = s.vol[j];
  slack |= slack_bond(r, p.horizon - 0.5 * p.h);
  if (isGreater(r, p.horizon - 0.5 * p.h)) v *= (p.horizon + 0.5 * p.h - r) / p.h;
  return 2. * r * infFn(s, r / p.horizon) * v * inv_scale;
}
__device__ __forceinline__ int list_entry(const DevTile& t, int gs, int j) {
  return t.lds ? (j - t.ws) * 16 : j - gs;
}
__device__ __forceinline__ uint64_t list_mix(uint64_t x) {  // splitmix64's finaliser
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

// hash of a tile's lists: degrees and entries of its nodes; a workgroup per tile
__global__ void __launch_bounds__(256) k_list_hash(DS s, const DevTile* tiles, unsigned long long* out) {
  __shared__ unsigned long long red[256 / WAVE];
  const DevTile t = tiles[blockIdx.x];
  const int gs = (int)s.P[t.pid].glob_start;
  unsigned long long h = 0;
  for (int l = threadIdx.x; l < t.te - t.ts; l += blockDim.x) {
    const int i = t.ts + l, n = s.deg[i];
    const int* c = s.col + s.sptr[i / WAVE] + i % WAVE;
    h += list_mix(((uint64_t)l << 34) + (uint64_t)n + 0x9e3779b97f4a7c15ull);
    for (int k = 0; k < n; k++)
      h += list_mix(((uint64_t)l << 34) ^ ((uint64_t)k << 17) ^ (uint64_t)list_entry(t, gs, c[(int64_t)k * WAVE]));
  }
  for (int o = WAVE / 2; o > 0; o >>= 1) h += __shfl_xor(h, o);
  if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = h;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// the lists of tiles[which[block]] from the PD neighbor lists
template <int DIM>
__global__ void __launch_bounds__(256) k_list_fill(DS s, MixedArgs m, const int* which, uint16_t* col16, float* wgt) {
  const DevTile t = m.tiles[which[blockIdx.x]];
  const DevParticle& p = s.P[t.pid];
  const int gs = (int)p.glob_start;
  const double inv_scale = 1. / particle_scale(s, p);
  for (int q = threadIdx.x; q < t.te - t.ts; q += blockDim.x) {
    const uint32_t ln = m.lnode[t.node + q];
    const int i = t.ts + (int)(ln & 0xffffu), n = (int)(ln >> 16);
    const int* c = s.col + s.sptr[i / WAVE] + i % WAVE;
    const int64_t at = t.data + m.lslice[t.slice + q / WAVE];
    for (int kb = 0; kb < n; kb += KB) {
      uint16_t* id = col16 + at + (int64_t)kb * WAVE + (q % WAVE) * KB;
      bool slack = false;
      unsigned id0 = 0;
      for (int k = kb; k < kb + KB; k++) {
        const int j = k < n ? c[(int64_t)k * WAVE] : -1;
        const unsigned e = k < n ? (unsigned)list_entry(t, gs, j) : t.lds ? (unsigned)(t.we - t.ws) * 16u : 0u;
        if (k == kb) id0 = e;
        id[k - kb] = (uint16_t)e;
        const double w = k < n ? bond_weight<DIM>(s, p, inv_scale, i, j, slack) : 0.;
        if (has_weights(s, m, t)) wgt[at + (int64_t)(k / 4) * WAVE * 4 + (q % WAVE) * 4 + k % 4] = (float)w;
      }
      if (slack && t.lds) id[0] = (uint16_t)(id0 | SLACK_BLOCK);
    }
  }
}

// whether the tiles' own lists equal the ones they are given (degrees and
// entries the same, weights, where they are read, within an ulp): diff[tile] is set where not
template <int DIM>
__global__ void __launch_bounds__(256) k_list_check(DS s, MixedArgs m, int* diff) {
  const DevTile t = m.tiles[blockIdx.x];
  const DevParticle& p = s.P[t.pid];
  const int gs = (int)p.glob_start;
  const double inv_scale = 1. / particle_scale(s, p);
  bool bad = false;
  for (int q = threadIdx.x; q < t.te - t.ts; q += blockDim.x) {
    const uint32_t ln = m.lnode[t.node + q];
    const int i = t.ts + (int)(ln & 0xffffu), n = (int)(ln >> 16);
    if (s.deg[i] != n) {
      bad = true;
      continue;
    }
    const int* c = s.col + s.sptr[i / WAVE] + i % WAVE;
    const int64_t at = t.data + m.lslice[t.slice + q / WAVE];
    const unsigned mask = t.lds ? SLACK_BLOCK - 1 : 0xffffu;
    for (int kb = 0; kb < n; kb += KB) {
      const uint16_t* id = m.col16 + at + (int64_t)kb * WAVE + (q % WAVE) * KB;
      bool slack = false;
      for (int k = kb; k < n && k < kb + KB; k++) {
        const int j = c[(int64_t)k * WAVE];
        const double w = bond_weight<DIM>(s, p, inv_scale, i, j, slack);
        bad |= (id[k - kb] & mask) != (unsigned)list_entry(t, gs, j);
        if (has_weights(s, m, t))
          bad |= !(fabs((double)m.wgt[at + (int64_t)(k / 4) * WAVE * 4 + (q % WAVE) * 4 + k % 4] - w) <=
                   0x1p-23 * fabs(w));
      }
      bad |= t.lds && ((id[0] & SLACK_BLOCK) != 0) != slack;
    }
  }
  if (bad) diff[blockIdx.x] = 1;
}

// the particles' constants (set-up); a workgroup each
__global__ void __launch_bounds__(256) k_mixed_part(DS s, int dim, PartConst* out) {
  __shared__ float red[256 / WAVE];
  const DevParticle& p = s.P[blockIdx.x];
  const int64_t gs = p.glob_start;
  double x = 0.;
  for (int64_t j = gs + threadIdx.x; j < p.glob_end; j += blockDim.x)
    for (int d = 0; d < dim; d++) x = fmax(x, fabs(s.xr[d][j] - s.xr[d][gs]));
  float mf = round_up(x);
  for (int o = WAVE / 2; o > 0; o >>= 1) mf = fmaxf(mf, __shfl_xor(mf, o));
  if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = mf;
  __syncthreads();
  if (threadIdx.x != 0 || p.glob_end <= gs) return;
  const double c = particle_scale(s, p);
  out[blockIdx.x] = PartConst{c, 1. / c, fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]))};
}

// the nodes' constant alpha terms (set-up)
__global__ void k_mixed_alpha(DS s, float* fa) {
  const int64_t i = gid();
  if (i >= s.N) return;
  const DevParticle& p = s.P[s.ptid[i]];
  fa[i] = (float)(2. * (15. * p.mat[1] / s.mx[i]) * particle_scale(s, p));
}

// copy of f of the nodes that take no PD force (save != 0: into buf, else
// back from it), around a standalone PD force pass; grid-stride
template <int DIM>
__global__ void k_noforce_copy(DS s, double* buf, int save) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = gid(); k < s.n_noforce; k += stride) {
    const int64_t i = s.noforce_nodes[k];
    for (int d = 0; d < DIM; d++) {
      if (save)
        buf[d * s.n_noforce + k] = s.f[d][i];
      else
        s.f[d][i] = buf[d * s.n_noforce + k];
    }
  }
}

}  // namespace pdem
