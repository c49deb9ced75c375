// Host-side launch plumbing shared by the per-equation translation units:
// argument block, grid shapes and the N -> NQ template dispatch.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "dg_kernels.h"

namespace canary {

enum Op { OP_VOLUME = 0, OP_FACE = 1, OP_UPDATE = 2, OP_STAGE = 3, OP_FACE_UPDATE = 4,
          OP_STAGE_PREP = 5 };

struct KArgs {
  void* rhs;
  const void* Q;
  void* Qout;
  const void* vgeo;
  const void* sgeo;
  const double* D;
  int64_t nreal, ntotal;
  const int64_t* vmapM;
  const int64_t* vmapP;
  const int64_t* bndy;
  double rka, rkb, dt;
  int advection;
  PhysParams phys;
  hipStream_t stream;
  const int32_t* pface;  // prepared face codes (OP_STAGE_PREP; vgeo, sgeo prepared too)
};

constexpr int kMaxN = 7;  // N = 1..7 compiled in

// The kernel families of a translation unit: the exact-order unit and the
// contracted unit (built with -ffp-contract=fast) hold every operation; the
// matrix-core unit the contracted unit's volume term and fused stages with
// the derivative contractions on the MFMA units (MfmaSweep).
enum Unit { UNIT_EXACT = 0, UNIT_FMA = 1, UNIT_MFMA = 2 };

inline int launch_status() {
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : 3 /*CANARY_ERR_LAUNCH*/;
}

// Element order of the in-place kernels (volumerhs, facerhs,
// updatesolution) and of the face + update fusion that follows a volumerhs:
// every launch of one of them walks the other way than the one before, so
// each starts on the elements the previous one touched last, whose lines the
// memory-side cache still holds (three-kernel stage at 3D N=4: 6.6% faster).
// The results of each element do not depend on the order.
inline int inplace_direction() {
  static std::atomic<unsigned> n{0};
  return (int)(n.fetch_add(1, std::memory_order_relaxed) & 1u);
}

// Block order of the in-place kernels.  A stage of them passes over the mesh
// several times.  Where its arrays nearly fit the 256 MB memory-side cache (210
// MB of them), a contiguous piece per XCD keeps each element on one XCD, and in
// its L2, through all passes; above that the runs of block_order are ahead.
// us for five stages of the three calls, in runs / in pieces: Euler 2D N=2 258^2
// (99 MB) 321 / 307, N=3 274^2 (183 MB) contracted 394 / 376, N=7 137^2 (159 MB)
// 420 / 404, total energy N=2 365^2 (198 MB) 514 / 492, shallow water N=7 137^2 320 /
// 308; N=1 548^2 (230 MB) 598 / 613, shallow water 552 / 576.
// facerhs_update reads and writes a second Q: N=2 258^2 485 / 464 us for two
// steps, N=3 274^2 (221 MB) 664 / 698.
constexpr int64_t kInplaceCache = 210000000;

template <class Phys, int NQ>
BlockOrder inplace_order(int64_t nblocks, const KArgs& a, bool second_q = false) {
  using S = Shape<Phys, NQ>;
  constexpr int DIM = Phys::DIM;
  constexpr int64_t bytes = 8 * (S::Np * (Phys::NS + Phys::NSR + DIM * DIM + 2) + S::NFN * (DIM + 3));
  const int64_t all = a.nreal * (bytes + (second_q ? 8 * S::Np * Phys::NS : 0));
  return block_order(nblocks, inplace_direction(), all > kInplaceCache);
}

// Element order of a ping-pong stage: the two Q buffers swap roles every
// stage, so their address order alternates and so does the direction.
inline int walk_back(const void* qin, const void* qout) {
  return (uintptr_t)qin > (uintptr_t)qout ? 1 : 0;
}

// Elements per workgroup of a stage.
//
// Small 2D meshes (at most kSmallBlocks blocks, eight workgroups a CU) take
// blocks of one wave: they wait for the latency of a workgroup, and one wave
// has no other to wait for at its barriers.  us for 4 steps, default against
// one wave: N=4 10 x 10 96 / 92, N=5 10 x 10 103 / 91, N=6 30 x 30 129 / 120,
// shallow water 40 x 40 N=4 123 / 108, N=6 156 / 143, total energy 40 x 40 N=4 133 /
// 116; above that size the default is ahead (N=5 50 x 50 149 / 161, N=6 170 / 174).
// Not where a SIMD would get more of these waves than a CU gets workgroups of
// the default: it is then one round of workgroups longer (2 steps at N=6, shallow
// water: 32 x 32, 1 and 1, default / one wave 64 / 61; 35 x 35, 1 and 2, 65 / 67; 36 x 36, 2
// and 2, 73 / 67; N=5 33 x 33, 1 and 2, 63 / 68).
// 3D N = 2 takes two elements, one wave, at every size: 20^3 103 / 88 us a step,
// 36^3 451 / 428, 53^3 1,405 / 1,374, prepared exact 1,513 / 1,463 (its volume and
// face kernels keep seven: facerhs 223 / 233).
constexpr int64_t kSmallBlocks = 8 * 256;

template <class Phys, int NQ, bool MFMA>
constexpr int stage_epw() {
  constexpr int Np = Shape<Phys, NQ>::Np;
  return Phys::DIM == 3 && NQ == 3 && !MFMA ? 64 / Np : default_epw<Np>();
}

// 0: no narrower block than the default
template <class Phys, int NQ>
constexpr int small_epw() {
  constexpr int Np = Shape<Phys, NQ>::Np;
  constexpr int w = Np <= 64 ? 64 / Np : 0;
  return Phys::DIM == 2 && w < default_epw<Np>() ? w : 0;
}

inline bool one_wave_blocks(int64_t nreal, int small, int epw) {
  auto rounds = [&](int e, int per_round) {
    const int64_t nb = (nreal + e - 1) / e;
    return (nb + per_round - 1) / per_round;
  };
  return nreal <= kSmallBlocks * small && rounds(small, 4 * 256) <= rounds(epw, 256);
}

template <class Phys, int NQ, int EPW, bool MFMA = false>
void launch_stage(const KArgs& a) {
  const int64_t nb = (a.nreal + EPW - 1) / EPW;
  constexpr int NT = FusedCfg<Phys, NQ, EPW>::NT;
  const BlockOrder order = block_order(nb, walk_back(a.Q, a.Qout));
  stage_kernel<Phys, NQ, EPW, MFMA><<<dim3((unsigned)(8 * order.chunk)), dim3(NT), 0, a.stream>>>(
      (double*)a.rhs, (const double*)a.Q, (double*)a.Qout, (const double*)a.vgeo,
      (const double*)a.sgeo, a.D, a.nreal, a.ntotal, a.vmapM, a.vmapP, a.bndy, a.rka, a.rkb,
      a.dt, order, a.phys, a.advection);
}

template <class Phys, int NQ, bool MFMA>
void launch_stage_sized(const KArgs& a) {
  constexpr int SMALL = small_epw<Phys, NQ>();
  constexpr int EPW = stage_epw<Phys, NQ, MFMA>();
  if constexpr (SMALL > 0)
    if (one_wave_blocks(a.nreal, SMALL, EPW)) return launch_stage<Phys, NQ, SMALL, MFMA>(a);
  launch_stage<Phys, NQ, EPW, MFMA>(a);
}

// Elements per workgroup of the contracted prepared 2D stage on large meshes:
// as many as 256 lanes hold.  Wider blocks read and write with fewer ragged
// ends and hold more of their neighbours; they pay where a stage moves more
// than the memory-side cache holds (from two million nodes on, 360 MB), below
// that the latency of a workgroup counts.  us per step, narrow against wide:
// 512^2 N=4 Euler 1,130 / 1,078, 500^2 N=2 421 / 402, 420^2 N=3 446 / 433,
// 250^2 N=7 595 / 577, shallow water 400^2 N=4 640 / 627, 250^2 N=7 532 / 522;
// smaller: 260^2 N=2 130 / 136, 150^2 N=7 220 / 225, 10 x 10 (50 stages) 241 /
// 267.  Kept narrow: N=1 (600^2: 271 / 292), the exact order, which needs more
// registers (200^2 N=7 454 / 473), 3D (32^3 N=4 1,051 / 1,085), and the
// reference arrays (shallow water 250^2 N=2 140 / 145).
template <class Phys, int NQ, int EPW>
constexpr int large_prep_epw() {
  constexpr int Np = Shape<Phys, NQ>::Np;
  return Phys::DIM == 2 && !Phys::EXACT && NQ > 2 && 256 / Np > EPW ? 256 / Np : EPW;
}
constexpr int64_t kLargePrepNodes = 2000000;

// The exact-order prepared 3D stage below N = 6 gathers early (see gather_late)
// on a mesh of at most one wave a SIMD: there no other wave covers the gather's
// latency, and its registers limit nothing.  us for two steps, late / early: N=1 8^3
// 95 / 87, 14^3 105 / 97, 20^3 (1,000 waves) 175 / 168, 27^3 176 / 180; N=2 9^3 90 / 83, 18^3 175 / 179;
// N=3 7^3 87 / 82, 10^3 103 / 98, 13^3 145 / 147; N=4 8^3 114 / 112, 11^3 164 / 167; N=5 5^3 86 / 84, 7^3
// 115 / 117.  (Over the reference arrays the late gathers are level or ahead there too.)
template <class Phys, int NQ, int EPW>
bool gather_early(int64_t nreal) {
  return (nreal + EPW - 1) / EPW * (FusedCfg<Phys, NQ, EPW>::NT / 64) <= 4 * 256;
}

template <class Phys, int NQ, int EPW, bool MFMA = false, bool EARLY = false>
void launch_stage_prep(const KArgs& a) {
  const int64_t nb = (a.nreal + EPW - 1) / EPW;
  constexpr int NT = FusedCfg<Phys, NQ, EPW>::NT;
  const BlockOrder order = block_order(nb, walk_back(a.Q, a.Qout));
  stage_prep_kernel<Phys, NQ, EPW, MFMA, EARLY><<<dim3((unsigned)(8 * order.chunk)), dim3(NT), 0, a.stream>>>(
      (double*)a.rhs, (const double*)a.Q, (double*)a.Qout, (const double*)a.vgeo,
      (const double*)a.sgeo, a.pface, a.D, a.nreal, a.ntotal, a.rka, a.rkb, a.dt, order,
      a.phys, a.advection);
}

// The prepared arrays hold no node heights: equation sets whose pressure
// needs them have no prepared stage.
template <class Phys, int NQ, bool MFMA = false>
void launch_stage_prep_if(const KArgs& a) {
  if constexpr (!NeedsY<Phys>::value) {
    constexpr int EPW = stage_epw<Phys, NQ, MFMA>();
    constexpr int SMALL = small_epw<Phys, NQ>();
    if constexpr (SMALL > 0)
      if (one_wave_blocks(a.nreal, SMALL, EPW)) return launch_stage_prep<Phys, NQ, SMALL, MFMA>(a);
    constexpr int BIG = large_prep_epw<Phys, NQ, EPW>();
    if constexpr (BIG > EPW)
      if (a.nreal * Shape<Phys, NQ>::Np >= kLargePrepNodes)
        return launch_stage_prep<Phys, NQ, BIG, MFMA>(a);
    if constexpr (Phys::DIM == 3 && gather_late<Phys, NQ>() && NQ < 7)
      if (gather_early<Phys, NQ, EPW>(a.nreal))
        return launch_stage_prep<Phys, NQ, EPW, MFMA, true>(a);
    launch_stage_prep<Phys, NQ, EPW, MFMA>(a);
  }
}

template <class Phys, int NQ, int EPW, bool MFMA>
void launch_volume(int64_t nb, const KArgs& a) {
  constexpr int NT = VolumeCfg<Phys, NQ, EPW>::NT;
  const BlockOrder order = inplace_order<Phys, NQ>(nb, a);
  volume_kernel<Phys, NQ, EPW, MFMA><<<dim3((unsigned)(8 * order.chunk)), dim3(NT), 0, a.stream>>>(
      (double*)a.rhs, (const double*)a.Q, (const double*)a.vgeo, a.D, a.nreal, order,
      a.phys);
}

// facerhs! reads rhs late (see late_rhs) where its workgroups do not all fit the
// 256 CUs' LDS at once with rhs read at the start.  Where they do, the smaller
// LDS gains nothing and the later load is waited for.  us for five stages of
// volumerhs! + facerhs! + updatesolution!, at the start / late, exact and
// contracted: N=1 27^3 (2,461 workgroups, 3,072 fit) 156 / 167 and 139 / 150,
// 33^3 235 / 228 and 205 / 199, 63^3 1,379 / 1,330 and 1,170 / 1,152; N=2 18^3 (833 of
// 1,280) 161 / 166 and 141 / 147, 22^3 215 / 206 and 185 / 174, 53^3 2,526 / 2,452 and
// 2,217 / 2,201; N=6 8^3 (512 of 768) 161 / 164 and 150 / 151, 12^3 355 / 345 and 305 /
// 287; N=7 8^3 (512 of 512) 177 / 177 and 152 / 153, 11^3 376 / 357 and 336 / 318.
template <class Phys, int NQ, int EPW>
bool late_rhs_pays(int64_t nb) {
  constexpr int64_t fit = 256 * (160 * 1024 / FusedCfg<Phys, NQ, EPW>::LDS);
  return nb > fit;
}

template <class Phys, int NQ, int EPW, bool LATE_R>
void launch_face_form(int64_t nb, const KArgs& a) {
  constexpr int NT = FusedCfg<Phys, NQ, EPW>::NT;
  const BlockOrder order = inplace_order<Phys, NQ>(nb, a);
  face_kernel<Phys, NQ, EPW, LATE_R><<<dim3((unsigned)(8 * order.chunk)), dim3(NT), 0, a.stream>>>(
      (double*)a.rhs, (const double*)a.Q, (const double*)a.vgeo, (const double*)a.sgeo, a.nreal,
      a.ntotal, a.vmapM, a.vmapP, a.bndy, order, a.phys);
}

template <class Phys, int NQ, int EPW>
void launch_face(int64_t nb, const KArgs& a) {
  if constexpr (late_rhs<Phys, NQ>())
    if (late_rhs_pays<Phys, NQ, EPW>(nb)) return launch_face_form<Phys, NQ, EPW, true>(nb, a);
  launch_face_form<Phys, NQ, EPW, false>(nb, a);
}

// Nonzero: the grid would not fit a launch.
template <class Phys, int NQ>
int launch_update(const KArgs& a) {
  const int64_t total = a.nreal * Shape<Phys, NQ>::Np;
  const int64_t nb = (total + 255) / 256;
  if (8 * ((nb + 7) / 8) > 0x7fffffffLL) return 1;
  const BlockOrder order = inplace_order<Phys, NQ>(nb, a);
  update_kernel<Phys, NQ><<<dim3((unsigned)(8 * order.chunk)), dim3(256), 0, a.stream>>>(
      (double*)a.rhs, (double*)a.Qout, (const double*)a.vgeo, a.nreal, a.rka, a.rkb, a.dt,
      a.advection, order);
  return 0;
}

template <class Phys, int NQ, int EPW>
void launch_face_update(int64_t nb, const KArgs& a) {
  constexpr int NT = FusedCfg<Phys, NQ, EPW>::NT;
  const BlockOrder order = inplace_order<Phys, NQ>(nb, a, true);
  face_update_kernel<Phys, NQ, EPW><<<dim3((unsigned)(8 * order.chunk)), dim3(NT), 0, a.stream>>>(
      (double*)a.rhs, (const double*)a.Q, (double*)a.Qout, (const double*)a.vgeo,
      (const double*)a.sgeo, a.nreal, a.ntotal, a.vmapM, a.vmapP, a.bndy, a.rka, a.rkb, a.dt,
      order, a.phys, a.advection);
}

// The operations a unit does not hold report CANARY_ERR_UNSUPPORTED.
template <class Phys, int NQ, int UNIT>
int launch(int op, const KArgs& a) {
  using S = Shape<Phys, NQ>;
  constexpr int EPW = default_epw<S::Np>();
  constexpr bool MFMA = UNIT == UNIT_MFMA;
  if (a.nreal <= 0) return 0;
  const int64_t nb = (a.nreal + EPW - 1) / EPW;
  if constexpr (UNIT != UNIT_EXACT) {
    if (op == OP_STAGE)
      launch_stage_sized<Phys, NQ, MFMA>(a);
    else if (op == OP_STAGE_PREP && !NeedsY<Phys>::value)
      launch_stage_prep_if<Phys, NQ, MFMA>(a);
    else if (op == OP_VOLUME)
      launch_volume<Phys, NQ, EPW, MFMA>(nb, a);
    else if (op == OP_FACE_UPDATE || op == OP_FACE || op == OP_UPDATE) {
      // no derivative contraction in these: the contracted unit holds them,
      // the matrix-core unit does not (each kernel lives in one unit)
      if constexpr (MFMA) {
        return 2 /*CANARY_ERR_UNSUPPORTED*/;
      } else {
        if (op == OP_FACE_UPDATE) launch_face_update<Phys, NQ, EPW>(nb, a);
        if (op == OP_FACE) launch_face<Phys, NQ, EPW>(nb, a);
        if (op == OP_UPDATE && launch_update<Phys, NQ>(a)) return 1 /*CANARY_ERR_ARG*/;
      }
    } else {
      return 2 /*CANARY_ERR_UNSUPPORTED*/;
    }
  } else {
    switch (op) {
      case OP_VOLUME:
        launch_volume<Phys, NQ, EPW, false>(nb, a);
        break;
      case OP_FACE:
        launch_face<Phys, NQ, EPW>(nb, a);
        break;
      case OP_UPDATE:
        if (launch_update<Phys, NQ>(a)) return 1 /*CANARY_ERR_ARG*/;
        break;
      case OP_STAGE:
        launch_stage_sized<Phys, NQ, false>(a);
        break;
      case OP_STAGE_PREP:
        if (NeedsY<Phys>::value) return 2 /*CANARY_ERR_UNSUPPORTED*/;
        launch_stage_prep_if<Phys, NQ>(a);
        break;
      case OP_FACE_UPDATE:
        launch_face_update<Phys, NQ, EPW>(nb, a);
        break;
      default:
        return 1 /*CANARY_ERR_ARG*/;
    }
  }
  return launch_status();
}

template <class Phys, int UNIT = UNIT_EXACT>
int dispatch(int op, int N, const KArgs& a) {
  switch (N) {
    case 1: return launch<Phys, 2, UNIT>(op, a);
    case 2: return launch<Phys, 3, UNIT>(op, a);
    case 3: return launch<Phys, 4, UNIT>(op, a);
    case 4: return launch<Phys, 5, UNIT>(op, a);
    case 5: return launch<Phys, 6, UNIT>(op, a);
    case 6: return launch<Phys, 7, UNIT>(op, a);
    case 7: return launch<Phys, 8, UNIT>(op, a);
  }
  return 2 /*CANARY_ERR_UNSUPPORTED*/;
}

// Read (and optionally clear) this translation unit's device error record.
inline int read_status(int64_t* info, int clear) {
  unsigned long long h[4] = {0, 0, 0, 0};
  if (hipMemcpyFromSymbol(h, HIP_SYMBOL(g_status), sizeof(h), 0, hipMemcpyDeviceToHost) != hipSuccess)
    return 3;
  if (clear && h[0] != 0) {
    unsigned long long z[4] = {0, 0, 0, 0};
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_status), z, sizeof(z), 0, hipMemcpyHostToDevice) != hipSuccess)
      return 3;
  }
  if (info)
    for (int i = 0; i < 4; ++i) info[i] = (int64_t)h[i];
  return (int)h[0];
}

}  // namespace canary

// The contracted-FP64 unit of an equation set (every operation), built with
// -ffp-contract=fast from a physics policy whose pressure avoids pow.
#define CANARY_DEFINE_FMA_STAGE(NAME, PHYS)                                       \
  extern "C" int canary_k_##NAME##_fma(int op, int N, const canary::KArgs* a) {  \
    return canary::dispatch<PHYS, canary::UNIT_FMA>(op, N, *a);                   \
  }                                                                               \
  extern "C" int canary_k_##NAME##_fma_status(int64_t* info, int clear) {        \
    return canary::read_status(info, clear);                                      \
  }

// The matrix-core unit: the contracted unit's volume term and fused stages
// with the derivative contractions on the MFMA units.
#define CANARY_DEFINE_MFMA_UNIT(NAME, PHYS)                                       \
  extern "C" int canary_k_##NAME##_mfma(int op, int N, const canary::KArgs* a) { \
    return canary::dispatch<PHYS, canary::UNIT_MFMA>(op, N, *a);                  \
  }                                                                               \
  extern "C" int canary_k_##NAME##_mfma_status(int64_t* info, int clear) {       \
    return canary::read_status(info, clear);                                      \
  }

#define CANARY_DEFINE_EQUATION(NAME, PHYS)                                        \
  extern "C" int canary_k_##NAME(int op, int N, const canary::KArgs* a) {        \
    return canary::dispatch<PHYS>(op, N, *a);                                     \
  }                                                                               \
  extern "C" int canary_k_##NAME##_status(int64_t* info, int clear) {            \
    return canary::read_status(info, clear);                                      \
  }
