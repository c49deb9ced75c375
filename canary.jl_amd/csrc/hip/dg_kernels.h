// Generic CDNA4 kernels of the nodal-DG right-hand side and LSRK update.
//
// Templated on the physics policy (phys.h), the number of 1-D nodes NQ = N+1
// and EPW, the number of elements one workgroup owns.  Threads map to
// (element slot, volume node) for volume work and to (element slot, face,
// face node) for face work; a workgroup is sized to a multiple of the
// 64-lane wavefront.
//
// Reference kernels these replace (behaviour, not structure):
//   knl_volumerhs!      examples/3d_kernels/euler3d_set2c.jl:366-486
//   knl_facerhs!        examples/3d_kernels/euler3d_set2c.jl:490-620
//   knl_updatesolution! examples/3d_kernels/euler3d_set2c.jl:624-639
//   (2D: euler2d_set2c.jl:318-524; SWE: shallow_water.jl:303-490)
//
// Evaluation order.  Each per-node result is accumulated in the order of
// the reference CPU kernels (euler3d_set2c.jl:144-358): rhs, then the
// buoyancy source, then the xi sweep n = 1..Nq, the eta sweep, the zeta
// sweep; then the face contributions in ascending face number; then the
// update Q + ((rkb*dt)*rhs)*MJI and rhs*rka.  With -ffp-contract=off and
// the correctly rounded pow of crpow.h (the oracle's pow is correctly
// rounded too) the exact-order kernels give the oracle's bits.
//
// Face terms are left in LDS and taken by each node's own thread, which knows
// its one to DIM face items from its indices: no atomics, and edge and corner
// nodes receive their face terms in ascending face order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "phys.h"
#include "mfma.h"

namespace canary {

constexpr int round64(int x) { return (x + 63) / 64 * 64; }
constexpr int ipow(int a, int b) { return b == 0 ? 1 : a * ipow(a, b - 1); }

template <class Phys, int NQ>
struct Shape {
  static constexpr int DIM = Phys::DIM;
  static constexpr int Np = ipow(NQ, DIM);
  static constexpr int Nfp = ipow(NQ, DIM - 1);
  static constexpr int NFACE = 2 * DIM;
  static constexpr int NFN = NFACE * Nfp;
};

// Elements per workgroup: smallest EPW whose round64(EPW*Np) keeps >= 90% of
// the lanes busy, else the best utilisation with at most 256 threads.
template <int Np>
constexpr int default_epw() {
  int best = 1;
  double bu = 0.0;
  for (int e = 1; e * Np <= 256 || e == 1; ++e) {
    double u = double(e * Np) / double(round64(e * Np));
    if (u >= 0.9) return e;
    if (u > bu + 1e-12) {
      bu = u;
      best = e;
    }
    if (e * Np > 256) break;
  }
  return best;
}

// Device-side error record of this translation unit:
// [code, face (1-based), element (1-based), offending value].
static __device__ unsigned long long g_status[4];

__device__ __forceinline__ void record_error(unsigned long long code, long long face,
                                             long long elem, long long value) {
  if (atomicCAS(&g_status[0], 0ull, code) == 0ull) {
    g_status[1] = (unsigned long long)face;
    g_status[2] = (unsigned long long)elem;
    g_status[3] = (unsigned long long)value;
  }
}

// Split a 1-based global node id into (element, node), 32-bit when it fits.
template <int Np>
__device__ __forceinline__ void split_id(int64_t id1, int64_t& elem, int& node) {
  const uint64_t id = (uint64_t)(id1 - 1);
  if ((id >> 32) == 0) {
    const uint32_t i32 = (uint32_t)id;
    elem = (int64_t)(i32 / (uint32_t)Np);
    node = (int)(i32 % (uint32_t)Np);
  } else {
    elem = (int64_t)(id / (uint64_t)Np);
    node = (int)(id % (uint64_t)Np);
  }
}

// XCD-aware block order: workgroups are dispatched round-robin over the 8
// XCDs, and the element blocks follow the Hilbert order, so runs of
// kXcdRun consecutive blocks are dealt to the XCDs in turn.  Within a run
// face neighbours share an L2; the XCDs together walk one window of
// 8*kXcdRun blocks, so memory sees one front per array instead of eight
// far-apart ones, and a neighbour in another XCD's run is in the memory-side
// cache.  Against one contiguous eighth of the mesh per XCD (us per stage):
// 512^2 2D N=4 prepared 246 -> 227, 32^3 N=4 prepared 221 -> 211, the three
// drop-in calls 451 -> 438 (runs of 16 or 256 blocks: within 2% of 64 either
// way).  The blocks past the last whole round of runs, and a launch of fewer
// than 16 runs per XCD, are split into contiguous pieces: such a mesh is in
// flight nearly as a whole, and the longer pieces only keep more neighbours
// together (one rank's 4,096 elements: 38.6 us against 39.3).  `deal` false:
// pieces alone (inplace_order in launch.h).
//
// A launch has 8*chunk workgroups and the map is one to one on them; the
// blocks beyond the mesh leave at once.  The host works out the order, the
// kernel spends a few scalar instructions on it (small meshes are bound by
// the latency of exactly such code).
//
// `reverse` walks the launch backwards.  Stages that ping-pong Q alternate
// the direction (the caller derives it from the buffer order, or the stage
// parity), so each stage starts on the elements the previous one touched
// last, whose lines the memory-side cache still holds (3D N=4, 32^3: 3.8%
// faster per stage).  Each element's result does not depend on the order.
constexpr uint32_t kXcdRun = 64;

struct BlockOrder {
  uint32_t chunk;  // blocks per XCD
  uint32_t dealt;  // of these, dealt in runs (a multiple of kXcdRun)
  uint32_t last;   // 8*chunk - 1 when walked backwards, else 0
};

inline BlockOrder block_order(int64_t nblocks, int reverse, bool deal = true) {
  BlockOrder o;
  o.chunk = (uint32_t)((nblocks + 7) / 8);
  o.dealt = !deal || o.chunk < 16 * kXcdRun ? 0 : o.chunk / kXcdRun * kXcdRun;
  o.last = reverse ? 8 * o.chunk - 1 : 0;
  return o;
}

__device__ __forceinline__ int64_t stage_block(uint32_t b, const BlockOrder& o) {
  b = o.last ? o.last - b : b;
  const uint32_t x = b & 7, i = b >> 3;
  const uint32_t run = (i / kXcdRun) * (8 * kXcdRun) + x * kXcdRun + i % kXcdRun;
  const uint32_t rest = 7 * o.dealt + x * (o.chunk - o.dealt) + i;
  return i < o.dealt ? run : rest;
}

// A pointer read from device memory (a row of a solve table) as one into
// global memory.  Without this its loads are flat: they count against the
// LDS counter too, so every LDS barrier and sweep waits for them, and the
// schedule of stage_body (loads left in flight over the sweeps) is lost.  A
// step of 16 precision-form solves: 3D 1,552 -> 1,502 us, 2D 192 -> 185; 48
// FP32 shallow-water solves, prepared, one launch: 240 -> 226.
// (Through an integer: a cast to the global address space and back is folded
// away before the compiler infers address spaces.)
template <class T>
__device__ __forceinline__ T* as_global(T* p) {
  return (T*)(__attribute__((address_space(1))) T*)(uintptr_t)p;
}

// a + x * y: in FP64 as the unit contracts it (the exact-order units do not),
// in FP32 fused.
__device__ __forceinline__ double mul_add(double x, double y, double a) { return a + x * y; }
__device__ __forceinline__ float mul_add(float x, float y, float a) { return fmaf(x, y, a); }
__device__ __forceinline__ double one_over(double x) { return 1.0 / x; }
__device__ __forceinline__ float one_over(float x) { return recip32(x); }

// ------------------------------------------------------------------ sweeps
// r[s] += sum_m D[m, i] F[m, j, k, s] (xi), then eta, then zeta, with the
// reference CPU order.  sF[d] points at the flux of direction d,
// laid out [s][node].
template <int DIM, int NQ, int NSR, class Real>
__device__ __forceinline__ void volume_sweeps(Real* r, const Real* sD, const Real* sF0,
                                              const Real* sF1, const Real* sF2, int n) {
  constexpr int Np = ipow(NQ, DIM);
  const int i = n % NQ;
  const int j = (n / NQ) % NQ;
  const int k = DIM == 3 ? n / (NQ * NQ) : 0;
  const int base_xi = n - i;                      // (0, j, k)
  const int base_eta = n - j * NQ;                // (i, 0, k)
  const int base_zeta = n - k * NQ * NQ;          // (i, j, 0)
#pragma unroll
  for (int s = 0; s < NSR; ++s) {
    Real a = r[s];
#pragma unroll
    for (int m = 0; m < NQ; ++m) a = mul_add(sD[m + NQ * i], sF0[s * Np + base_xi + m], a);
#pragma unroll
    for (int m = 0; m < NQ; ++m) a = mul_add(sD[m + NQ * j], sF1[s * Np + base_eta + m * NQ], a);
    if (DIM == 3) {
#pragma unroll
      for (int m = 0; m < NQ; ++m) a = mul_add(sD[m + NQ * k], sF2[s * Np + base_zeta + m * NQ * NQ], a);
    }
    r[s] = a;
  }
}

// r[s] += sum_m D[m, i_dir] F[..m..][s] along direction DIR only (same per-state
// accumulation order as volume_sweeps when called for DIR = 0, 1, 2 in turn).
template <int DIM, int NQ, int NSR, class Real, int DIR>
__device__ __forceinline__ void volume_sweep_dir(Real* r, const Real* sD, const Real* sF, int n) {
  constexpr int Np = ipow(NQ, DIM);
  constexpr int STRIDE = DIR == 0 ? 1 : (DIR == 1 ? NQ : NQ * NQ);
  const int idx = DIR == 0 ? n % NQ : (DIR == 1 ? (n / NQ) % NQ : n / (NQ * NQ));
  const int base = n - idx * STRIDE;
#pragma unroll
  for (int s = 0; s < NSR; ++s) {
    Real a = r[s];
#pragma unroll
    for (int m = 0; m < NQ; ++m) a = mul_add(sD[m + NQ * idx], sF[s * Np + base + m * STRIDE], a);
    r[s] = a;
  }
}

// ------------------------------------------------------------ face terms
// A face item is one face node `fi` (= f*Nfp + fn) of element e.  Its work
// is split in three steps so that a kernel can issue the loads early and
// consume them later: face_meta (normal, sMJ, maps, bc), face_gather (the
// P-side state from Q) and face_finish (wall state, pressure, Rusanov flux,
// times sMJ -- the amount the reference subtracts from rhs).
template <class Phys>
struct FaceItem {
  using Real = typename Phys::Real;
  Real nrm[Phys::DIM];
  Real sMJ;
  Real qP[Phys::NS];
  Real yP;  // height of the P node (equation sets whose pressure needs it)
  int64_t eP;
  int64_t idM, idP, bcode;  // map and bc entries as loaded (face_load_maps)
  int vidM;  // -1: no contribution (an error was recorded)
  int vidP;
  int bc;
};

// Barrier for threads that exchange data through LDS only: waits for LDS
// traffic (lgkmcnt) but leaves global loads in flight across the barrier.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Volume node (0-based) of face node fn of face f: the canonical face mask
// of src/mesh.jl:978-982 -- dimension f/2 held at its first (even f) or last
// (odd f) index, the other dimensions in column-major order.  vmapM[:,f,e]
// is always Np*(e-1) + this + 1 (src/mesh.jl:994).
template <int DIM, int NQ>
__device__ __forceinline__ int canon_vid(int f, int fn) {
  constexpr int N = NQ - 1;
  const int fe = (f & 1) * N;
  if (DIM == 2) return (f >> 1) == 0 ? fe + NQ * fn : fn + NQ * fe;
  const int a = fn % NQ, b = fn / NQ;
  switch (f >> 1) {
    case 0: return fe + NQ * a + NQ * NQ * b;
    case 1: return a + NQ * fe + NQ * NQ * b;
    default: return a + NQ * b + NQ * NQ * fe;
  }
}

// face_meta in parts: face_load_maps and face_load_geo issue the loads (no
// use of their values, so a kernel can issue more loads behind them),
// face_resolve checks the maps and bc and splits the node ids.
//
// A null vmapM stands for the canonical face mask (the only vmapM that
// src/mesh.jl builds): the M-side id is computed, and the map load re-reads
// the vmapP entry instead (a cache hit, no HBM bytes), so both forms run one
// instruction sequence in one kernel.
template <class Phys, int NQ>
__device__ __forceinline__ void face_load_maps(FaceItem<Phys>& it,
                                               const int64_t* __restrict__ vmapM,
                                               const int64_t* __restrict__ vmapP,
                                               const int64_t* __restrict__ bndy, int64_t e,
                                               int fi) {
  using S = Shape<Phys, NQ>;
  constexpr int DIM = Phys::DIM;
  const int f = fi / S::Nfp;
  const size_t fo = (size_t)fi + (size_t)S::NFN * (size_t)e;
  const bool canon = vmapM == nullptr;
  const int64_t rawM = (canon ? vmapP : vmapM)[fo];
  it.idP = vmapP[fo];
  it.idM = canon ? (int64_t)S::Np * e + canon_vid<DIM, NQ>(f, fi - f * S::Nfp) + 1 : rawM;
  it.bcode = bndy[f + S::NFACE * e];
}

// normal and sMJ of face item fi of element e, NSG words a record
template <class Phys, int NQ, int NSG>
__device__ __forceinline__ void face_load_geo(FaceItem<Phys>& it,
                                              const typename Phys::Real* __restrict__ sgeo,
                                              int64_t e, int fi) {
  constexpr int DIM = Phys::DIM, NFN = Shape<Phys, NQ>::NFN;
  const typename Phys::Real* sg = sgeo + (size_t)NSG * ((size_t)fi + (size_t)NFN * (size_t)e);
#pragma unroll
  for (int c = 0; c < DIM; ++c) it.nrm[c] = sg[c];
  it.sMJ = sg[DIM];
}

// The maps are split and selected without branching on them (a load whose
// value is first used under a branch is moved under it by the compiler, and
// then waiting for it waits for every load issued before); errors are
// recorded in the reference's order of checks: vmapM, then vmapP of an
// interior face, then the bc code.
template <class Phys, int NQ>
__device__ __forceinline__ void face_resolve(FaceItem<Phys>& it, int64_t e, int fi,
                                             int64_t ntotal) {
  using S = Shape<Phys, NQ>;
  constexpr int Np = S::Np;
  const int f = fi / S::Nfp;
  const int64_t idM = it.idM, idP = it.idP, bc = it.bcode;
  const int64_t nodes = ntotal * (int64_t)Np;
  const bool okM = idM >= 1 && idM <= nodes;
  const bool okP = idP >= 1 && idP <= nodes;
  const bool interior = bc == 0;
  const bool good = okM && (bc == 1 || (interior && okP));
  int64_t eP, eM;
  int vP, vM;
  split_id<Np>(okP ? idP : 1, eP, vP);
  split_id<Np>(okM ? idM : 1, eM, vM);
  it.bc = (int)bc;
  it.eP = good && interior ? eP : 0;
  it.vidP = good && interior ? vP : 0;
  it.vidM = good ? vM : -1;  // -1: no contribution
  if (!good) {
    if (!okM)
      record_error(5 /*CANARY_ERR_VMAP*/, f + 1, e + 1, idM);
    else if (interior)
      record_error(5 /*CANARY_ERR_VMAP*/, f + 1, e + 1, idP);
    else
      record_error(4 /*CANARY_ERR_BC*/, f + 1, e + 1, bc);
  }
}

template <class Phys, int NQ>
__device__ __forceinline__ void face_meta(FaceItem<Phys>& it,
                                          const typename Phys::Real* __restrict__ sgeo,
                                          const int64_t* __restrict__ vmapM,
                                          const int64_t* __restrict__ vmapP,
                                          const int64_t* __restrict__ bndy, int64_t e, int fi,
                                          int64_t ntotal) {
  face_load_maps<Phys, NQ>(it, vmapM, vmapP, bndy, e, fi);
  face_load_geo<Phys, NQ, Phys::NSGEO>(it, sgeo, e, fi);
  face_resolve<Phys, NQ>(it, e, fi, ntotal);
}

// ---------------------------------------------------- prepared geometry
// The compact arrays canary_prepare_geometry builds once from the reference
// ones (vmapM the canonical face mask, every face in the orientation
// `mappings` supports, MJI = 1 / MJ, elemtobndy 0 or 1 -- all checked
// there):
//   pvgeo (Np, DIM*DIM + 1, nelem): metric terms and MJ (no MJI, no x, y, z)
//   psgeo (DIM + 1, Nfp, NFACE, nelem): normal and sMJ (no vMJI)
//   pface int32 (NFACE, nelem): -1 for a wall face (bc 1), else
//         NFACE * eP + fP, the neighbour element and its face (0-based):
//         vmapP[fn, f, e] = Np * eP + fmask[fn, fP] + 1 (src/mesh.jl:994-995)
template <class Phys>
struct Prepared {
  static constexpr int DIM = Phys::DIM;
  static constexpr int NV = DIM * DIM + 1;  // pvgeo fields
  static constexpr int NSG = DIM + 1;       // psgeo fields
};

// face_load_maps over the prepared arrays: the face code goes to idP and is
// turned into node ids by face_decode_resolve once it has arrived.
template <class Phys, int NQ>
__device__ __forceinline__ void face_load_code(FaceItem<Phys>& it,
                                               const int32_t* __restrict__ pface, int64_t e,
                                               int fi) {
  using S = Shape<Phys, NQ>;
  it.idP = pface[fi / S::Nfp + S::NFACE * e];
}

// face_decode + face_resolve over the prepared arrays, without building the
// 1-based node ids and splitting them again: the code (an int32, as loaded)
// gives the neighbour and its face directly.  The values are those the two
// steps give (the M side is always in range; a neighbour beyond ntotal is
// the same vmap error, with the same payload).
template <class Phys, int NQ>
__device__ __forceinline__ void face_decode_resolve(FaceItem<Phys>& it, int64_t e, int fi,
                                                    int64_t ntotal) {
  using S = Shape<Phys, NQ>;
  constexpr int DIM = Phys::DIM;
  const int f = fi / S::Nfp, fn = fi - f * S::Nfp;
  const int32_t code = (int32_t)it.idP;
  const bool wall = code < 0;
  const int32_t eP = wall ? 0 : code / S::NFACE;
  const int fP = wall ? f : code - eP * S::NFACE;
  const int vP = canon_vid<DIM, NQ>(fP, fn);
  const bool ok = wall || (int64_t)eP < ntotal;
  it.bc = wall ? 1 : 0;
  it.eP = wall || !ok ? 0 : eP;
  it.vidP = wall || !ok ? 0 : vP;
  it.vidM = ok ? canon_vid<DIM, NQ>(f, fn) : -1;  // -1: no contribution
  if (!ok) record_error(5 /*CANARY_ERR_VMAP*/, f + 1, e + 1, (int64_t)S::Np * eP + vP + 1);
}

// The height y of node v of element e (vgeo field iY), for the equation
// sets whose pressure needs it.
template <class Phys, int NQ>
__device__ __forceinline__ typename Phys::Real node_y(const typename Phys::Real* __restrict__ vgeo,
                                                      int64_t e, int v) {
  if constexpr (NeedsY<Phys>::value) {
    constexpr int Np = Shape<Phys, NQ>::Np;
    return vgeo[(size_t)Phys::NVGEO * Np * (size_t)e + (size_t)Phys::iY * Np + v];
  } else {
    return typename Phys::Real(0);
  }
}

template <class Phys, int NQ>
__device__ __forceinline__ void face_gather(FaceItem<Phys>& it,
                                            const typename Phys::Real* __restrict__ Q,
                                            const typename Phys::Real* __restrict__ vgeo) {
  constexpr int Np = Shape<Phys, NQ>::Np, NS = Phys::NS;
  if (it.vidM >= 0 && it.bc == 0) {
    const typename Phys::Real* qe = Q + (size_t)NS * Np * (size_t)it.eP;
#pragma unroll
    for (int s = 0; s < NS; ++s) it.qP[s] = qe[it.vidP + Np * s];
    it.yP = node_y<Phys, NQ>(vgeo, it.eP, it.vidP);
  }
}

// face_gather with a load on every lane: items without a P-side state
// (invalid, wall, bad map) read node 0 of element e_safe, which is in bounds,
// and leave qP to face_finish.
template <class Phys, int NQ>
__device__ __forceinline__ void face_gather_any(FaceItem<Phys>& it,
                                                const typename Phys::Real* __restrict__ Q,
                                                const typename Phys::Real* __restrict__ vgeo,
                                                bool valid, int64_t e_safe) {
  constexpr int Np = Shape<Phys, NQ>::Np, NS = Phys::NS;
  const bool ok = valid && it.vidM >= 0 && it.bc == 0;
  const typename Phys::Real* qe = Q + (size_t)NS * Np * (size_t)(ok ? it.eP : e_safe);
  const int v = ok ? it.vidP : 0;
  typename Phys::Real g[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) g[s] = qe[v + Np * s];
  const typename Phys::Real y = node_y<Phys, NQ>(vgeo, ok ? it.eP : e_safe, v);
  if (ok) {
#pragma unroll
    for (int s = 0; s < NS; ++s) it.qP[s] = g[s];
    it.yP = y;
  }
}

// M-side state through qm_at(s, node) and pm_at(node, qM); out[NSR].
template <class Phys, class QM, class PMF>
__device__ __forceinline__ int face_finish(FaceItem<Phys>& it, const PhysParams& p, QM qm_at,
                                           PMF pm_at, typename Phys::Real* out) {
  using Real = typename Phys::Real;
  constexpr int NS = Phys::NS;
  if (it.vidM < 0) return -1;
  Real qM[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) qM[s] = qm_at(s, it.vidM);
  const Real PM = pm_at(it.vidM, qM);
  Real PP = 0;
  if (it.bc == 0) {
    if (Phys::B_FROM_M) it.qP[NS - 1] = qm_at(NS - 1, it.vidP);
    PP = Phys::HAS_P ? pressure_at<Phys>(it.qP, it.yP, p) : Real(0);
  } else {
    Phys::reflect(qM, PM, it.nrm, it.qP, PP);
  }
  Phys::face_flux(qM, PM, it.qP, PP, it.nrm, it.sMJ, p, out);
  return it.vidM;
}

// All three steps at once.
template <class Phys, int NQ, class QM, class PMF>
__device__ __forceinline__ int face_contribution(const typename Phys::Real* __restrict__ Q,
                                                 const typename Phys::Real* __restrict__ vgeo,
                                                 const typename Phys::Real* __restrict__ sgeo,
                                                 const int64_t* __restrict__ vmapM,
                                                 const int64_t* __restrict__ vmapP,
                                                 const int64_t* __restrict__ bndy, int64_t e,
                                                 int fi, int64_t ntotal, const PhysParams& p,
                                                 QM qm_at, PMF pm_at, typename Phys::Real* out) {
  FaceItem<Phys> it;
  face_meta<Phys, NQ>(it, sgeo, vmapM, vmapP, bndy, e, fi, ntotal);
  face_gather<Phys, NQ>(it, Q, vgeo);
  return face_finish<Phys>(it, p, qm_at, pm_at, out);
}

// The face terms of volume node n, subtracted from r in ascending face order
// (the order facerhs! applies them: it walks the faces in turn, and a node
// lies on at most one face of each pair 2d, 2d+1): with vmapM the canonical
// face mask, the term of face item f*Nfp + fn lands on node canon_vid(f, fn),
// so the node owner finds its one to DIM items from its own indices.  sC:
// the items' terms [fi][s]; sV: their node ids, NOVID where an item has no
// term (an error was recorded).
template <int DIM, int NQ, int NSR, class Real, class VidT>
__device__ __forceinline__ void face_terms_at_node(Real* r, const Real* sC, const VidT* sV, int n,
                                                   VidT novid) {
  constexpr int Nfp = ipow(NQ, DIM - 1);
  const int i = n % NQ, j = (n / NQ) % NQ, k = DIM == 3 ? n / (NQ * NQ) : 0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int idx = d == 0 ? i : (d == 1 ? j : k);
    if (idx == 0 || idx == NQ - 1) {
      const int f = 2 * d + (idx == 0 ? 0 : 1);
      const int fn = DIM == 2 ? (d == 0 ? j : i)
                              : (d == 0 ? j + NQ * k : (d == 1 ? i + NQ * k : i + NQ * j));
      const int fi = f * Nfp + fn;
      if (sV[fi] != novid) {
#pragma unroll
        for (int s = 0; s < NSR; ++s) r[s] = r[s] - sC[fi * NSR + s];
      }
    }
  }
}

// The same for any vmapM, by the whole workgroup (EPW elements of which the
// first nv are there, node n of element `slot` in r, items in sV and sC as
// above with BUF words an element).  The items of each face pair leave their
// number at their node in a table (tab: TSTR words of Real an element, free
// until r is stored), and the node owner takes one term per pair, in
// ascending order.  Where two items of a pair name one node, which no
// numbering of a face does, the owners look through all items instead, which
// is right for every map and several times the work.  Bound by its barriers and
// LDS round trips, little beside the rest of a launch: facerhs! at 3D N=7 16^3, us,
// canonical map 70, every face reversed 71 (searched 285); N=4 25^3 83 and 86 (183).
template <int DIM, int NQ, int EPW, int NT, int NSR, int BUF, int TSTR, class Real, class VidT>
__device__ __forceinline__ void face_terms_any_map(Real* r, const Real* sB, const VidT* sV,
                                                   Real* tab, int* sFlag, VidT novid, int nv,
                                                   int slot, int n, bool valid) {
  constexpr int Np = ipow(NQ, DIM), Nfp = ipow(NQ, DIM - 1), NFN = 2 * DIM * Nfp;
  static_assert(sizeof(Real) * NSR >= sizeof(int) * DIM, "the table fits rhs's place");
  auto table = [&](int sl) { return reinterpret_cast<int*>(tab + sl * TSTR); };
  if (valid) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) table(slot)[d * Np + n] = -1;
  }
  lds_barrier();
  for (int item = threadIdx.x; item < nv * NFN; item += NT) {
    const int sl = EPW == 1 ? 0 : item / NFN, fi = item - sl * NFN;
    if (sV[item] != novid) table(sl)[fi / (2 * Nfp) * Np + sV[item]] = fi;
  }
  lds_barrier();
  for (int item = threadIdx.x; item < nv * NFN; item += NT) {
    const int sl = EPW == 1 ? 0 : item / NFN, fi = item - sl * NFN;
    if (sV[item] != novid && table(sl)[fi / (2 * Nfp) * Np + sV[item]] != fi) *sFlag = 2;
  }
  int fi[DIM];
  if (valid) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) fi[d] = table(slot)[d * Np + n];
  }
  lds_barrier();  // the table is read (r may take its place) and checked
  if (valid) {
    const Real* sC = sB + slot * BUF;
    if (*sFlag == 2) {
#pragma unroll 1
      for (int k = 0; k < NFN; ++k)
        if (sV[slot * NFN + k] == (VidT)n) {
#pragma unroll
          for (int s = 0; s < NSR; ++s) r[s] = r[s] - sC[k * NSR + s];
        }
    } else {
#pragma unroll
      for (int d = 0; d < DIM; ++d)
        if (fi[d] >= 0) {
#pragma unroll
          for (int s = 0; s < NSR; ++s) r[s] = r[s] - sC[fi[d] * NSR + s];
        }
    }
  }
}

// ================================================================ kernels
template <class Phys, int NQ, int EPW>
struct VolumeCfg {
  using S = Shape<Phys, NQ>;
  static constexpr int NT = round64(EPW * S::Np);
};

// MFMA: the derivative contractions on the matrix cores (MfmaSweep), in
// place in sF, then r + xi + eta + zeta at each node; else volume_sweeps.
template <class Phys, int NQ, int EPW, bool MFMA = false>
__global__ __launch_bounds__((VolumeCfg<Phys, NQ, EPW>::NT)) void volume_kernel(
    double* __restrict__ rhs, const double* __restrict__ Q, const double* __restrict__ vgeo,
    const double* __restrict__ D, int64_t nreal, BlockOrder order, PhysParams p) {
  using S = Shape<Phys, NQ>;
  constexpr int Np = S::Np, DIM = S::DIM, NS = Phys::NS, NSR = Phys::NSR, NV = Phys::NVGEO;
  __shared__ double sD[NQ * NQ];
  __shared__ double sF[DIM][EPW][NSR * Np];
  const int64_t blk = stage_block(blockIdx.x, order);
  if (blk * EPW >= nreal) return;  // whole workgroup leaves together
  const int t = threadIdx.x;
  const int slot = t / Np, n = t - slot * Np;
  const int64_t e = blk * EPW + slot;
  const bool valid = slot < EPW && e < nreal;
  if (t < NQ * NQ) sD[t] = D[t];
  double r[NSR];
  if (valid) {
    double q[NS];
    const double* qe = Q + (size_t)NS * Np * (size_t)e;
#pragma unroll
    for (int s = 0; s < NS; ++s) q[s] = qe[n + Np * s];
    const double* vg = vgeo + (size_t)NV * Np * (size_t)e;
    double met[DIM * DIM];
#pragma unroll
    for (int c = 0; c < DIM * DIM; ++c) met[c] = vg[n + Np * c];
    const double MJ = vg[n + Np * Phys::iMJ];
    const double P = Phys::HAS_P ? pressure_at<Phys>(q, node_y<Phys, NQ>(vgeo, e, n), p) : 0.0;
    double F[DIM][NSR];
    Phys::volume_flux(q, P, met, MJ, p, F);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      // MFMA: each direction line by line (MfmaSweep)
      const int w = MFMA ? MfmaSweep<DIM, NQ, NSR>::slot_of(d, n) : n;
#pragma unroll
      for (int s = 0; s < NSR; ++s) sF[d][slot][s * Np + w] = F[d][s];
    }
    const double* re = rhs + (size_t)NS * Np * (size_t)e;
#pragma unroll
    for (int s = 0; s < NSR; ++s) r[s] = re[n + Np * s];
    Phys::source(q, MJ, p, r);
  }
  lds_barrier();
  if constexpr (MFMA) {
    const int nv = nreal - blk * EPW < EPW ? (int)(nreal - blk * EPW) : EPW;
    mfma_sweeps<DIM, NQ, NSR, VolumeCfg<Phys, NQ, EPW>::NT, EPW, DIM>(
        &sF[0][0][0], EPW * NSR * Np, NSR * Np, nv, sD);
    lds_barrier();
    if (valid) {
      int w[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d) w[d] = MfmaSweep<DIM, NQ, NSR>::slot_of(d, n);
#pragma unroll
      for (int s = 0; s < NSR; ++s) {
        double a = r[s];
#pragma unroll
        for (int d = 0; d < DIM; ++d) a = a + sF[d][slot][s * Np + w[d]];
        r[s] = a;
      }
    }
  } else if (valid) {
    volume_sweeps<DIM, NQ, NSR>(r, sD, sF[0][slot], sF[DIM > 1 ? 1 : 0][slot],
                                sF[DIM > 2 ? 2 : 0][slot], n);
  }
  if (valid) {
    double* re = rhs + (size_t)NS * Np * (size_t)e;
#pragma unroll
    for (int s = 0; s < NSR; ++s) re[n + Np * s] = r[s];
  }
}


template <class Phys, int NQ>
__global__ __launch_bounds__(256) void update_kernel(double* __restrict__ rhs,
                                                     double* __restrict__ Q,
                                                     const double* __restrict__ vgeo,
                                                     int64_t nreal, double rka, double rkb,
                                                     double dt, int advection,
                                                     BlockOrder order) {
  using S = Shape<Phys, NQ>;
  constexpr int Np = S::Np, NS = Phys::NS, NSR = Phys::NSR, NV = Phys::NVGEO;
  const int64_t total = nreal * Np;
  const double bdt = rkb * dt;
  {
    const int64_t g = stage_block(blockIdx.x, order) * 256 + threadIdx.x;
    if (g >= total) return;
    const int64_t e = g / Np;
    const int n = (int)(g - e * Np);
    const double MJI = vgeo[n + Np * (Phys::iMJI + (size_t)NV * e)];
    double* qe = Q + (size_t)NS * Np * e;
    double* re = rhs + (size_t)NS * Np * e;
    double uu = 0.0, vv = 0.0;
    if (Phys::HAS_ADVECTION && advection) {
      const double Ht = qe[n + Np * 2] + qe[n + Np * 3];
      uu = qe[n] / Ht;
      vv = qe[n + Np] / Ht;
    }
#pragma unroll
    for (int s = 0; s < NSR; ++s) {
      const double r = re[n + Np * s];
      qe[n + Np * s] = qe[n + Np * s] + bdt * r * MJI;
      re[n + Np * s] = r * rka;
    }
    if (Phys::HAS_ADVECTION && advection) {
      const double Ht = qe[n + Np * 2] + qe[n + Np * 3];
      qe[n] = Ht * uu;
      qe[n + Np] = Ht * vv;
    }
  }
}

// --------------------------------------------------------- fused stage
// One LSRK stage of EPW elements per workgroup: volume term, face terms and
// update in one pass over HBM.  Reads Qin (own + neighbour traces), writes
// Qout; rhs in place.
//
// Schedule (per workgroup):
//   1. each thread issues the loads of its first face item (maps, bc; unless
//      gather_late its normal and sMJ), of D and of its volume node's Q,
//      metric terms and rhs, before it uses any of them;
//   2. volume fluxes in registers; the P-side gather of the face item before
//      them, as soon as its map has arrived, or (gather_late) after them;
//   3. the xi/eta/zeta sweeps run through one flux buffer in LDS while the
//      gathers are in flight (barriers fence LDS only, so loads stay
//      outstanding across them); rhs accumulates in registers;
//   4. face fluxes -> LDS, taken by each node's thread in ascending face order;
//   5. update: Qout = Q + ((rkb*dt)*rhs)*MJI, rhs *= rka, to LDS;
//   6. the block's Qout and rhs written out in storage order.
// RES: room for rhs beside the face terms.
template <class Phys, int NQ, int EPW, bool RES = true>
struct FusedCfg {
  // vidM of each face node fits a byte up to Np = 255, else a short
  using VidT = typename std::conditional<(Shape<Phys, NQ>::Np < 256), uint8_t, uint16_t>::type;
  using S = Shape<Phys, NQ>;
  using Real = typename Phys::Real;
  static constexpr int NT = round64(EPW * S::Np);
  static constexpr int FLUX = S::Np;                       // per state, one direction
  static constexpr int FACE = S::NFN + (RES ? S::Np : 0);   // face terms + rhs per state
  static constexpr int FLUX_ = RES ? FLUX : 0;              // (late_rhs: no fluxes)
  static constexpr int BUF = (FLUX_ > FACE ? FLUX_ : FACE) * Phys::NSR;
  // LDS carve-up (bytes, each piece 16-byte aligned)
  static constexpr int a16(int b) { return (b + 15) / 16 * 16; }
  static constexpr int OFF_D = 0;
  static constexpr int OFF_Q = OFF_D + a16(sizeof(Real) * NQ * NQ);
  static constexpr int OFF_P = OFF_Q + a16(sizeof(Real) * EPW * Phys::NS * S::Np);
  static constexpr int OFF_B = OFF_P + a16(sizeof(Real) * EPW * (Phys::HAS_P ? S::Np : 1));
  static constexpr int OFF_V = OFF_B + a16(sizeof(Real) * EPW * BUF);
  static constexpr int OFF_F = OFF_V + a16(sizeof(VidT) * EPW * S::NFN);  // one flag word
  static constexpr int LDS = OFF_F + 16;
};

// When a stage issues its face items' geometry and P-side gathers: before the
// volume fluxes, so that they have the longest time to arrive, or (LATE) after
// them, in flight over the sweeps, so that their registers are not live with
// the metric terms.  LATE pays where registers limit the waves that fit: the
// exact-order 3D kernels (32^3 N=4, reference arrays: 1,422 -> 1,377 us a step;
// N=7: 1,342 -> 1,235) and the contracted ones from N = 6 on; the contracted
// ones below are faster early (N=5: 1,042 against 1,058), as is 2D (10 x 10
// meshes wait for latency alone: 240 against 269 us for 50 stages), and as the
// exact prepared stage is on a mesh of one wave a SIMD (gather_early, launch.h).
//
// 3D N = 6 has 343 nodes in six waves: at 96 VGPRs five waves fit a SIMD and
// three workgroups a CU, above that two.  It is built for that (stage_waves),
// with the maps read after the fluxes too (MAPS_LATE) and rhs left in LDS
// over the face phase; without these it spills.  23^3 stage 348 -> 304 us,
// prepared loop exact 1,619 -> 1,416, contracted 1,302 -> 1,137.
template <class Phys, int NQ>
constexpr bool gather_late() {
  if constexpr (Phys::DIM == 3)
    return Phys::EXACT || NQ >= 7;
  else
    return false;
}

template <class Phys, int NQ>
constexpr int stage_waves() {  // waves a SIMD must hold
  return Phys::DIM == 3 && NQ == 7 ? 5 : 1;
}

// facerhs! alone at these 3D orders may read rhs after the face terms and
// leave its results in Q's place, which nothing reads any more by then: without
// rhs beside the face terms a fifth (N=1) to a third (N=6, 7) less LDS, so more
// workgroups fit a CU (late_rhs_pays in launch.h has the line).
// N = 3, 4, 5 are level or 2-3% faster with rhs read at the start, as 2D is.
template <class Phys, int NQ>
constexpr bool late_rhs() {
  return Phys::DIM == 3 && (NQ <= 3 || NQ >= 7);
}

// One fused stage of the EPW-element block starting at e0, computed by NT
// threads (NT >= the volume nodes of the block).  `lds` holds
// FusedCfg::LDS bytes.  Each thread's first face item is loaded with its node's
// arrays (the rest, where there are more items than threads, afterwards).
// VOLUME = false leaves the volume term out (face terms + update only: the
// opt-in facerhs_update, after a separate volumerhs); vgeo is then read for
// MJI alone and D is not read.  UPDATE = false (with VOLUME = false) is
// facerhs! alone: rhs -= face terms, Q untouched, neither vgeo nor Qout read;
// LATE_R: rhs read after the face terms (late_rhs).  EARLY: gathers before the
// volume fluxes whatever gather_late says.
template <class Phys, int NQ, int EPW, int NT, bool VOLUME = true, bool UPDATE = true,
          bool PREP = false, bool MFMA = false, bool LATE_R = false, bool EARLY = false>
__device__ __forceinline__ void stage_body(
    char* __restrict__ lds, typename Phys::Real* __restrict__ rhs,
    const typename Phys::Real* __restrict__ Qin, typename Phys::Real* __restrict__ Qout,
    const typename Phys::Real* __restrict__ vgeo, const typename Phys::Real* __restrict__ sgeo,
    const double* __restrict__ D, int64_t e0, int64_t nreal, int64_t ntotal,
    const int64_t* __restrict__ vmapM, const int64_t* __restrict__ vmapP,
    const int64_t* __restrict__ bndy, double rka, double rkb, double dt, const PhysParams& p,
    int advection = 0) {
  using S = Shape<Phys, NQ>;
  static_assert(!LATE_R || (!VOLUME && !UPDATE), "facerhs! alone");
  using C = FusedCfg<Phys, NQ, EPW, !LATE_R>;
  using Real = typename Phys::Real;
  constexpr int Np = S::Np, DIM = S::DIM, NS = Phys::NS, NSR = Phys::NSR;
  constexpr int NV = PREP ? Prepared<Phys>::NV : Phys::NVGEO;
  constexpr int NFN = S::NFN, Nfp = S::Nfp;
  static_assert(!PREP || (VOLUME && UPDATE), "prepared arrays: the whole stage only");
  static_assert(!NeedsY<Phys>::value || !PREP,
                "a pressure that needs y: the reference arrays hold it");
  // prepared arrays: psgeo in `sgeo`, the face codes in `vmapP`'s place
  const int32_t* __restrict__ pface = reinterpret_cast<const int32_t*>(vmapP);
  // Face items per thread loaded with the node's arrays.  More than one costs
  // registers.  The code over them stays loops of one: written straight out, the
  // compiler moves the item's loads under `if (fval)` (10 x 10 loop 231.7 -> 235.4 us).
  constexpr int KP = 1;
  constexpr bool LATE = VOLUME && gather_late<Phys, NQ>() && !EARLY;
  constexpr bool N6 = stage_waves<Phys, NQ>() > 1;
  constexpr bool MAPS_LATE = LATE && !PREP && N6;
  constexpr bool STAGE_R = (!VOLUME && !LATE_R) || (VOLUME && N6);  // rhs waits in LDS for the face terms
  constexpr int NSG = PREP ? Prepared<Phys>::NSG : Phys::NSGEO;
  constexpr int BUF = C::BUF;
  using VidT = typename C::VidT;
  constexpr VidT NOVID = (VidT)~(VidT)0;
  static_assert(NT >= EPW * Np, "one volume node per thread");
  static_assert(!MFMA || (VOLUME && std::is_same<Real, double>::value),
                "matrix-core contractions: FP64 volume term");
  Real* sD = reinterpret_cast<Real*>(lds + C::OFF_D);
  Real* sQ = reinterpret_cast<Real*>(lds + C::OFF_Q);  // [EPW][NS*Np]
  Real* sP = reinterpret_cast<Real*>(lds + C::OFF_P);  // [EPW][Np]
  Real* sB = reinterpret_cast<Real*>(lds + C::OFF_B);  // [EPW][BUF]
  VidT* sV = reinterpret_cast<VidT*>(lds + C::OFF_V);  // [EPW][NFN]
  int* sFlag = reinterpret_cast<int*>(lds + C::OFF_F);  // a non-canonical M-side node seen

  Real* sR = LATE_R ? sQ : sB + NFN * NSR;  // rhs results, RSTR words an element
  constexpr int RSTR = LATE_R ? NS * Np : BUF;

  const int t = threadIdx.x;
  const int slot = EPW == 1 ? 0 : t / Np, n = t - slot * Np;
  const bool valid = EPW == 1 ? t < Np : slot < EPW && e0 + slot < nreal;

  // 1. issue the loads of the block before any of them is used: the face
  //    items' maps and bc (t, t + NT, ...), D, the node's Q, metric terms and
  //    rhs -- one memory round trip instead of one per kind.  The loads are
  //    unconditional (lanes without work read in-bounds element e0, node 0,
  //    and ignore it): a load under a branch makes every later wait count
  //    for the path without it, i.e. wait for everything.
  FaceItem<Phys> fit[KP];
  bool fval[KP];
  int fsl[KP], ffi[KP];
#pragma unroll
  for (int k = 0; k < KP; ++k) {
    const int item = t + k * NT;
    fsl[k] = EPW == 1 ? 0 : item / NFN;
    fval[k] = item < EPW * NFN && (EPW == 1 || e0 + fsl[k] < nreal);
    fsl[k] = fval[k] ? fsl[k] : 0;
    ffi[k] = fval[k] ? item - fsl[k] * NFN : 0;
    if constexpr (PREP)
      face_load_code<Phys, NQ>(fit[k], pface, e0 + fsl[k], ffi[k]);
    else if constexpr (!MAPS_LATE)
      face_load_maps<Phys, NQ>(fit[k], vmapM, vmapP, bndy, e0 + fsl[k], ffi[k]);
    if constexpr (!LATE) face_load_geo<Phys, NQ, NSG>(fit[k], sgeo, e0 + fsl[k], ffi[k]);
  }
  double dval = 0.0;
  if constexpr (VOLUME) dval = D[t < NQ * NQ ? t : 0];
  // keep the map loads ahead of the node loads: waiting for the maps then
  // leaves the node loads in flight (the wait counter is in issue order)
  __builtin_amdgcn_sched_barrier(0);
  const int sl0 = valid ? slot : 0, nl = valid ? n : 0;
  const int64_t el = e0 + sl0;
  Real q[NS], met[DIM * DIM], r[NSR];
  const Real* qe = Qin + (size_t)NS * Np * (size_t)e0 + (sl0 * NS * Np + nl);
#pragma unroll
  for (int s = 0; s < NS; ++s) q[s] = qe[Np * s];
  const Real* vg = (VOLUME || UPDATE)
                       ? vgeo + (size_t)NV * Np * (size_t)e0 + (sl0 * NV * Np + nl)
                       : nullptr;
  // the node's height, for a pressure that needs it (loaded with the rest)
  const Real ynode = NeedsY<Phys>::value ? node_y<Phys, NQ>(vgeo, el, nl) : Real(0);
  Real MJ = 0;
  if constexpr (VOLUME) {
#pragma unroll
    for (int c = 0; c < DIM * DIM; ++c) met[c] = vg[Np * c];
    MJ = vg[Np * Phys::iMJ];
  }
  const Real* re = rhs + (size_t)NS * Np * (size_t)e0 + (sl0 * NS * Np + nl);
  if constexpr (!LATE_R) {
#pragma unroll
    for (int s = 0; s < NSR; ++s) r[s] = re[Np * s];
  }
  // maps checked as soon as they arrive and the P-side gathers issued
  // (unconditionally, as above: lanes without an item check the item
  // they loaded, e0's first face node, which some lane owns anyway)
  auto gather = [&]() {
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      if constexpr (LATE && !MAPS_LATE)
        face_load_geo<Phys, NQ, NSG>(fit[k], sgeo, e0 + fsl[k], ffi[k]);
      if constexpr (PREP)
        face_decode_resolve<Phys, NQ>(fit[k], e0 + fsl[k], ffi[k], ntotal);
      else
        face_resolve<Phys, NQ>(fit[k], e0 + fsl[k], ffi[k], ntotal);
      face_gather_any<Phys, NQ>(fit[k], Qin, vgeo, fval[k], e0);
    }
  };
  if constexpr (!LATE) gather();

  if (VOLUME && t < NQ * NQ) sD[t] = (Real)dval;
  if (!PREP && t == 0) *sFlag = 0;  // read after the face terms, barriers later
  // 2. volume fluxes
  Real Fv[DIM][NSR];
  if (valid) {
#pragma unroll
    for (int s = 0; s < NS; ++s) sQ[slot * NS * Np + s * Np + n] = q[s];
    const Real P = Phys::HAS_P ? pressure_at<Phys>(q, ynode, p) : Real(0);
    if constexpr (Phys::HAS_P) sP[slot * Np + n] = P;
    if constexpr (VOLUME) {
      Phys::volume_flux(q, P, met, MJ, p, Fv);
      Phys::source(q, MJ, p, r);
    }
  }
  if constexpr (LATE) {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MAPS_LATE) {
#pragma unroll
      for (int k = 0; k < KP; ++k) {
        face_load_maps<Phys, NQ>(fit[k], vmapM, vmapP, bndy, e0 + fsl[k], ffi[k]);
        face_load_geo<Phys, NQ, NSG>(fit[k], sgeo, e0 + fsl[k], ffi[k]);
      }
    } else {
      gather();
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  Real MJI = 0;
  if constexpr (UPDATE && !PREP && !MAPS_LATE) MJI = vg[Np * Phys::iMJI];
  // 3. sweeps, one direction at a time through one flux buffer
#pragma unroll
  for (int d = 0; d < (VOLUME ? DIM : 0); ++d) {
    if (d > 0) lds_barrier();  // the previous direction's fluxes are consumed
    // MFMA: the direction line by line (MfmaSweep)
    const int w = MFMA ? MfmaSweep<DIM, NQ, NSR>::slot_of(d, n) : n;
    if (valid) {
#pragma unroll
      for (int s = 0; s < NSR; ++s) sB[slot * BUF + s * Np + w] = Fv[d][s];
    }
    lds_barrier();
    if constexpr (MFMA) {
      // the direction's contractions in place in sB, then added by the node
      const int nvb = nreal - e0 < EPW ? (int)(nreal - e0) : EPW;
      mfma_sweeps<DIM, NQ, NSR, NT, EPW, 1>(reinterpret_cast<double*>(sB), 0, BUF, nvb,
                                            reinterpret_cast<const double*>(sD));
      lds_barrier();
      if (valid) {
#pragma unroll
        for (int s = 0; s < NSR; ++s) r[s] = r[s] + sB[slot * BUF + s * Np + w];
      }
    } else if (valid) {
      const Real* b = sB + slot * BUF;
      if (d == 0) volume_sweep_dir<DIM, NQ, NSR, Real, 0>(r, sD, b, n);
      if (d == 1) volume_sweep_dir<DIM, NQ, NSR, Real, (DIM > 1 ? 1 : 0)>(r, sD, b, n);
      if (d == 2) volume_sweep_dir<DIM, NQ, NSR, Real, (DIM > 2 ? 2 : 0)>(r, sD, b, n);
    }
    if constexpr (MAPS_LATE) {
      if (d == 0) {
        __builtin_amdgcn_sched_barrier(0);
        gather();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  lds_barrier();  // fluxes consumed (and Q, P staged): face terms take their place
  if constexpr (STAGE_R) {
    if (valid) {
#pragma unroll
      for (int s = 0; s < NSR; ++s) sB[slot * BUF + NFN * NSR + s * Np + n] = r[s];
    }
  }
  // 4. face fluxes: M side from LDS, P side gathered
  bool noncanon = false;  // an item whose M-side node is not the canonical one
  auto pm_of = [&](int sl, int v, const Real* qm) -> Real {
    if constexpr (Phys::HAS_P)
      return sP[sl * Np + v];
    else
      return Phys::pressure(qm, p);
  };
#pragma unroll
  for (int k = 0; k < KP; ++k) {
    if (!fval[k]) continue;
    const int sl = fsl[k], fi = ffi[k];
    auto qm_at = [&](int s, int v) { return sQ[sl * NS * Np + s * Np + v]; };
    auto pm_at = [&](int v, const Real* qm) { return pm_of(sl, v, qm); };
    Real c[NSR];
    const int vid = face_finish<Phys>(fit[k], p, qm_at, pm_at, c);
    if constexpr (!PREP) noncanon |= vid >= 0 && vid != canon_vid<DIM, NQ>(fi / Nfp, fi % Nfp);
    sV[sl * NFN + fi] = vid < 0 ? NOVID : (VidT)vid;
#pragma unroll
    for (int s = 0; s < NSR; ++s) sB[sl * BUF + fi * NSR + s] = c[s];
  }
  for (int item = t + KP * NT; item < EPW * NFN; item += NT) {
    const int sl = EPW == 1 ? 0 : item / NFN, fi = item - sl * NFN;
    if (EPW > 1 && e0 + sl >= nreal) continue;
    auto qm_at = [&](int s, int v) { return sQ[sl * NS * Np + s * Np + v]; };
    auto pm_at = [&](int v, const Real* qm) { return pm_of(sl, v, qm); };
    Real c[NSR];
    int vid;
    if constexpr (PREP) {
      FaceItem<Phys> it;
      face_load_code<Phys, NQ>(it, pface, e0 + sl, fi);
      face_load_geo<Phys, NQ, NSG>(it, sgeo, e0 + sl, fi);
      face_decode_resolve<Phys, NQ>(it, e0 + sl, fi, ntotal);
      face_gather<Phys, NQ>(it, Qin, vgeo);
      vid = face_finish<Phys>(it, p, qm_at, pm_at, c);
    } else {
      vid = face_contribution<Phys, NQ>(Qin, vgeo, sgeo, vmapM, vmapP, bndy, e0 + sl, fi, ntotal, p,
                                        qm_at, pm_at, c);
      noncanon |= vid >= 0 && vid != canon_vid<DIM, NQ>(fi / Nfp, fi % Nfp);
    }
    sV[sl * NFN + fi] = vid < 0 ? NOVID : (VidT)vid;
#pragma unroll
    for (int s = 0; s < NSR; ++s) sB[sl * BUF + fi * NSR + s] = c[s];
  }
  if (!PREP && NT > 64 && noncanon) *sFlag = 1;
  if constexpr (LATE_R) {
#pragma unroll
    for (int s = 0; s < NSR; ++s) r[s] = re[Np * s];
  }
  lds_barrier();
  // 5. each node's thread takes its own face terms in ascending face order
  //    (with the canonical face mask, always so over the prepared arrays, it
  //    finds them from its indices; over the reference arrays, a workgroup
  //    with any other vmapM makes a table), then updates.
  //    Shallow water with `advection` keeps the velocity: u = Hu / (h + b)
  //    before the update, Hu = (h + b) u after it (shallow_water.jl:274-297).
  bool any_map = false;
  if constexpr (!PREP) {
    // (one wave needs no word in LDS for it: 10 x 10 loop 231.4 -> 230.1 us)
    any_map = NT == 64 ? __any(noncanon) : __builtin_amdgcn_readfirstlane(*sFlag) != 0;
    if (any_map) {
      const int nv = nreal - e0 < EPW ? (int)(nreal - e0) : EPW;
      if constexpr (STAGE_R) {
        Real x[NSR];
        Real* const xs = sB + slot * BUF + NFN * NSR + n;
        if (valid) {
#pragma unroll
          for (int s = 0; s < NSR; ++s) x[s] = xs[s * Np];
        }
        lds_barrier();  // the table takes rhs's place
        face_terms_any_map<DIM, NQ, EPW, NT, NSR, BUF, RSTR>(x, sB, sV, sR, sFlag, NOVID, nv,
                                                             slot, n, valid);
        if (valid) {
#pragma unroll
          for (int s = 0; s < NSR; ++s) xs[s * Np] = x[s];
        }
        // back through LDS, not kept in registers: live over this branch it
        // would cost every launch eight of them
        asm volatile("" ::: "memory");
      } else {
        face_terms_any_map<DIM, NQ, EPW, NT, NSR, BUF, RSTR>(r, sB, sV, sR, sFlag, NOVID, nv,
                                                             slot, n, valid);
      }
    }
  }
  if (valid) {
    if constexpr (STAGE_R) {
#pragma unroll
      for (int s = 0; s < NSR; ++s) r[s] = sB[slot * BUF + NFN * NSR + s * Np + n];
    }
    if (!any_map)
      face_terms_at_node<DIM, NQ, NSR>(r, sB + slot * BUF, sV + slot * NFN, n, NOVID);
    if constexpr (UPDATE) {
      // prepared arrays hold no MJI: the reference's is 1 ./ MJ (IEEE division;
      // FP32: refined estimate)
      if constexpr (PREP) MJI = one_over(MJ);
      if constexpr (MAPS_LATE) MJI = vg[Np * Phys::iMJI];
      const Real bdt = (Real)(rkb * dt);
      const Real ka = (Real)rka;
      Real* qn = sQ + slot * NS * Np + n;
      Real uu = 0, vv = 0;
      if (Phys::HAS_ADVECTION && advection) {
        const Real Ht = qn[Np * 2] + qn[Np * 3];
        uu = qn[0] / Ht;
        vv = qn[Np] / Ht;
      }
#pragma unroll
      for (int s = 0; s < NSR; ++s) {
        Real& qq = qn[s * Np];
        const Real rs = r[s];
        qq = mul_add(bdt * rs, MJI, qq);
        r[s] = rs * ka;
      }
      if (Phys::HAS_ADVECTION && advection) {
        const Real Ht = qn[Np * 2] + qn[Np * 3];
        qn[0] = Ht * uu;
        qn[Np] = Ht * vv;
      }
    }
  }
  if (valid) {
#pragma unroll
    for (int s = 0; s < NSR; ++s) sR[slot * RSTR + s * Np + n] = r[s];
  }
  lds_barrier();
  // 6. the block's results leave LDS in storage order: consecutive lanes
  //    write consecutive words, so every wave writes whole lines (a store per
  //    state from the node owners writes Np-word runs that start and end
  //    inside lines; 2D N=4: 7-9% slower).  Non-temporal stores: nothing
  //    reads these lines again in this stage, and keeping them out of L2
  //    leaves room for the Q lines the face gathers reuse (3D N=4: 600 fewer
  //    bytes fetched per element, 3% faster).
  const int nv = nreal - e0 < EPW ? (int)(nreal - e0) : EPW;
  if constexpr (UPDATE) {
    Real* qo = Qout + (size_t)NS * Np * (size_t)e0;
    for (int i = t; i < nv * NS * Np; i += NT) __builtin_nontemporal_store(sQ[i], &qo[i]);
  }
  {
    Real* ro = rhs + (size_t)NS * Np * (size_t)e0;
    for (int i = t; i < nv * NSR * Np; i += NT) {
      const int sl = EPW == 1 ? 0 : i / (NSR * Np), j = i - sl * (NSR * Np);
      __builtin_nontemporal_store(sR[sl * RSTR + j], &ro[sl * (NS * Np) + j]);
    }
  }
}

template <class Phys, int NQ, int EPW, bool MFMA = false>
__global__ __launch_bounds__((FusedCfg<Phys, NQ, EPW>::NT), (stage_waves<Phys, NQ>())) void stage_kernel(
    double* __restrict__ rhs, const double* __restrict__ Qin, double* __restrict__ Qout,
    const double* __restrict__ vgeo, const double* __restrict__ sgeo,
    const double* __restrict__ D, int64_t nreal, int64_t ntotal,
    const int64_t* __restrict__ vmapM, const int64_t* __restrict__ vmapP,
    const int64_t* __restrict__ bndy, double rka, double rkb, double dt,
    BlockOrder order, PhysParams p, int advection) {
  using C = FusedCfg<Phys, NQ, EPW>;
  __shared__ __attribute__((aligned(16))) char lds[C::LDS];
  const int64_t blk = stage_block(blockIdx.x, order);
  const int64_t e0 = blk * EPW;
  if (e0 >= nreal) return;  // whole workgroup leaves together
  stage_body<Phys, NQ, EPW, C::NT, true, true, false, MFMA>(
      lds, rhs, Qin, Qout, vgeo, sgeo, D, e0, nreal, ntotal, vmapM, vmapP, bndy, rka, rkb, dt, p,
      advection);
}

// The fused stage over the prepared arrays (see Prepared): the same
// arithmetic and order, fewer bytes.
template <class Phys, int NQ, int EPW, bool MFMA = false, bool EARLY = false>
__global__ __launch_bounds__((FusedCfg<Phys, NQ, EPW>::NT), (stage_waves<Phys, NQ>())) void stage_prep_kernel(
    double* __restrict__ rhs, const double* __restrict__ Qin, double* __restrict__ Qout,
    const double* __restrict__ pvgeo, const double* __restrict__ psgeo,
    const int32_t* __restrict__ pface, const double* __restrict__ D, int64_t nreal,
    int64_t ntotal, double rka, double rkb, double dt, BlockOrder order, PhysParams p,
    int advection) {
  using C = FusedCfg<Phys, NQ, EPW>;
  __shared__ __attribute__((aligned(16))) char lds[C::LDS];
  const int64_t blk = stage_block(blockIdx.x, order);
  const int64_t e0 = blk * EPW;
  if (e0 >= nreal) return;  // whole workgroup leaves together
  stage_body<Phys, NQ, EPW, C::NT, true, true, true, MFMA, false, EARLY>(
      lds, rhs, Qin, Qout, pvgeo, psgeo, D, e0, nreal, ntotal, nullptr,
      reinterpret_cast<const int64_t*>(pface), nullptr, rka, rkb, dt, p, advection);
}

// facerhs! alone (rhs -= sMJ * Rusanov flux of Q): the fused stage body with
// its volume term and update switched off, so the face terms get the same
// schedule (every load issued first, nodal Q and pressure staged in LDS for
// the M side, non-temporal rhs stores) and the same bits.  vgeo is read only
// by equation sets whose pressure needs the node height (else it may be
// null).
template <class Phys, int NQ, int EPW, bool LATE_R>
__global__ __launch_bounds__((FusedCfg<Phys, NQ, EPW>::NT)) void face_kernel(
    double* __restrict__ rhs, const double* __restrict__ Q, const double* __restrict__ vgeo,
    const double* __restrict__ sgeo, int64_t nreal, int64_t ntotal,
    const int64_t* __restrict__ vmapM, const int64_t* __restrict__ vmapP,
    const int64_t* __restrict__ bndy, BlockOrder order, PhysParams p) {
  using C = FusedCfg<Phys, NQ, EPW, !LATE_R>;
  __shared__ __attribute__((aligned(16))) char lds[C::LDS];
  const int64_t blk = stage_block(blockIdx.x, order);
  const int64_t e0 = blk * EPW;
  if (e0 >= nreal) return;  // whole workgroup leaves together
  stage_body<Phys, NQ, EPW, C::NT, false, false, false, false, LATE_R>(
      lds, rhs, Q, nullptr, vgeo, sgeo, nullptr, e0, nreal, ntotal, vmapM, vmapP, bndy, 0.0, 0.0,
      0.0, p);
}

// facerhs! + updatesolution! of one stage in one pass (the volume term was
// added to rhs by volume_kernel before): Qin -> Qout, rhs in place.
template <class Phys, int NQ, int EPW>
__global__ __launch_bounds__((FusedCfg<Phys, NQ, EPW>::NT)) void face_update_kernel(
    double* __restrict__ rhs, const double* __restrict__ Qin, double* __restrict__ Qout,
    const double* __restrict__ vgeo, const double* __restrict__ sgeo, int64_t nreal,
    int64_t ntotal, const int64_t* __restrict__ vmapM, const int64_t* __restrict__ vmapP,
    const int64_t* __restrict__ bndy, double rka, double rkb, double dt,
    BlockOrder order, PhysParams p, int advection) {
  using C = FusedCfg<Phys, NQ, EPW>;
  __shared__ __attribute__((aligned(16))) char lds[C::LDS];
  const int64_t blk = stage_block(blockIdx.x, order);
  const int64_t e0 = blk * EPW;
  if (e0 >= nreal) return;  // whole workgroup leaves together
  stage_body<Phys, NQ, EPW, C::NT, false>(lds, rhs, Qin, Qout, vgeo, sgeo, nullptr, e0,
                                                   nreal, ntotal, vmapM, vmapP, bndy, rka, rkb,
                                                   dt, p, advection);
}

}  // namespace canary
