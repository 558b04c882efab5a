// Phase B on CDNA4: one wavefront per column, levels across lanes.
//
// Level k of a column lives in lane k % 64 of register chunk k / 64; the
// kernel is compiled for 1 to kSedMaxChunks chunks and a launch takes the
// fewest that hold its levels; columns of more levels run one lane each.  The column couplings of the
// reference's sedimentation (src/module_mp_tempo_main.F90:590-727) become
// wavefront primitives:
//   top-down fill of a fall-speed profile (:1768-1789 and species variants)
//       -> ballot of the levels holding mass, lowest set bit at or above
//          each lane, value fetched by a lane permute;
//   CFL substep count and ktop -> wavefront max reductions;
//   one flux-form substep (:1516-1559) -> every level at once, the flux
//          from the level above by a one-lane shift (all fluxes of a
//          substep use the fields at its start, so the levels are
//          independent within it).
// Every per-level operand is staged through LDS: a block takes one column
// group of the column-tiled scratch (kScrW columns whose levels are
// contiguous), reads it as one contiguous run and transposes it to
// (column, level) rows that one wavefront reads with unit stride; all planes
// of a species are requested together.
//
// The arithmetic per level is the serial kernel's, operation for operation,
// so both give identical results.
#pragma once

#include <cstring>
#include <type_traits>

#include "tempo_step.hpp"

namespace tempo {

constexpr unsigned kFlagsChanged = 1u << 31;  // of a thread's copy of a point's flags: to be written back
constexpr int kSedCols = kScrW;           // columns (wavefronts) per block: one scratch column group
constexpr int kSedSlots = 8;              // LDS planes staged at once
constexpr int kSedMaxChunks = 4;          // register chunks of 64 levels of the largest form
constexpr int kSedMaxLevels = 64 * kSedMaxChunks;
constexpr int kSedChunks = 2;             // chunks of the adjoint's column kernels
constexpr int kSedLevels = 64 * kSedChunks;

// Staged values are kept as the scratch holds them: 4 bytes in the FP32
// step (the sedimentation widens them in registers, and rounds the
// tendencies once on the way back, as a store from FP64 would), 8 bytes
// otherwise.  Half the LDS lets twice the blocks share a CU; at 160 levels,
// where eight FP64 planes take 82 KB, it decides between one block and four.
template <class R>
using SedStage = typename std::conditional<std::is_same<Sd_t<R>, float>::value, float, double>::type;
// The kernel's types: X of masses, tendencies and speeds while they sediment,
// V of level geometry and raw speeds, E of the staged planes.  A dual working
// type runs on the values alone (the tangent-free forward of an adjoint), or,
// with kTan, on duals throughout (the tangent-linear step).
template <class R, bool kTan>
struct SedTypes {
  using X = typename std::conditional<kTan, W_t<R>, double>::type;
  using V = typename std::conditional<kTan, R, S_t<R>>::type;
  using E = typename std::conditional<kTan, W_t<R>, SedStage<R>>::type;
};
// LDS row of one column, in stage elements: at least nz, and an odd multiple
// of 8 (4-byte elements) or 4 (8-byte), so that the 8 columns x 8 (4) levels
// that a wavefront (half one) writes at a time fall in 64 different banks
template <class E>
__host__ __device__ constexpr int sed_row(int nz) {
  return ((nz + int(32 / sizeof(E)) - 1) / int(32 / sizeof(E)) | 1) * int(32 / sizeof(E));
}
template <class E>
__host__ __device__ constexpr size_t sed_lds_bytes(int nz) {
  return size_t(kSedSlots) * kSedCols * sed_row<E>(nz) * sizeof(E);
}

namespace wv {
__device__ __forceinline__ int lane() { return int(threadIdx.x & 63u); }
// Data-parallel-primitive moves between lanes: one VALU instruction per 32
// bits, against an LDS permute (and its wait) for a general shuffle.  The
// sedimentation's substeps are chains of such moves (131,072 uneven columns
// of up to 22 substeps: 1.02 -> 0.86 ms).
template <int ctrl, int rows = 0xf, class T>
__device__ __forceinline__ T dpp(T old, T x) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "32- or 64-bit values");
  if constexpr (sizeof(T) == 4) {
    const int r = __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, x), ctrl, rows, 0xf, false);
    return __builtin_bit_cast(T, r);
  } else {
    const long long o = __builtin_bit_cast(long long, old), v = __builtin_bit_cast(long long, x);
    const unsigned lo = unsigned(__builtin_amdgcn_update_dpp(int(o), int(v), ctrl, rows, 0xf, false));
    const unsigned hi = unsigned(__builtin_amdgcn_update_dpp(int(o >> 32), int(v >> 32), ctrl, rows, 0xf, false));
    return __builtin_bit_cast(T, (static_cast<unsigned long long>(hi) << 32) | lo);
  }
}
// x of lane l (the same l in every lane)
template <class T>
__device__ __forceinline__ T read_lane(T x, int l) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
  } else {
    const long long v = __builtin_bit_cast(long long, x);
    const unsigned lo = unsigned(__builtin_amdgcn_readlane(int(v), l));
    const unsigned hi = unsigned(__builtin_amdgcn_readlane(int(v >> 32), l));
    return __builtin_bit_cast(T, (static_cast<unsigned long long>(hi) << 32) | lo);
  }
}
template <int ctrl, int rows = 0xf, class T>
__device__ __forceinline__ Dual<T> dpp(Dual<T> old, Dual<T> x) {
  return {dpp<ctrl, rows>(old.v, x.v), dpp<ctrl, rows>(old.d, x.d)};
}
template <class T>
__device__ __forceinline__ Dual<T> read_lane(Dual<T> x, int l) {
  return {read_lane(x.v, l), read_lane(x.d, l)};
}
// maximum (of non-negative values) and bitwise or over the wavefront: row
// shifts by 1, 2, 4, 8, then the rows' last lanes broadcast upwards
__device__ __forceinline__ int imax(int v) {
  v = max(v, dpp<0x111>(0, v));
  v = max(v, dpp<0x112>(0, v));
  v = max(v, dpp<0x114>(0, v));
  v = max(v, dpp<0x118>(0, v));
  v = max(v, dpp<0x142, 0xa>(0, v));
  v = max(v, dpp<0x143, 0xc>(0, v));
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ unsigned uor(unsigned v) {
  v |= dpp<0x111>(0u, v);
  v |= dpp<0x112>(0u, v);
  v |= dpp<0x114>(0u, v);
  v |= dpp<0x118>(0u, v);
  v |= dpp<0x142, 0xa>(0u, v);
  v |= dpp<0x143, 0xc>(0u, v);
  return unsigned(__builtin_amdgcn_readlane(int(v), 63));
}
// value of x at level k (per lane), chunks held in x[]
template <class T, int CH>
__device__ __forceinline__ T at_level(const T (&x)[CH], int k) {
  T v = T(0);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const T t = __shfl(x[j], k & 63, 64);
    if ((k >> 6) == j) v = t;
  }
  return v;
}
// ... at a level that is the same in every lane
template <class T, int CH>
__device__ __forceinline__ T at_uniform(const T (&x)[CH], int k) {
  T v = read_lane(x[0], k & 63);
#pragma unroll
  for (int j = 1; j < CH; ++j)
    if ((k >> 6) == j) v = read_lane(x[j], k & 63);
  return v;
}
// value of x at level k+1 for every lane's level k in chunk j (0 above the top chunk)
template <class T, int CH>
__device__ __forceinline__ T above(const T (&x)[CH], int j) {
  T top = T(0);
  if (j + 1 < CH) top = read_lane(x[j + 1 < CH ? j + 1 : j], 0);
  return dpp<0x130>(top, x[j]);  // whole-wavefront shift: lane l takes lane l + 1
}
}  // namespace wv

// the value of a stored number as a double (the staging carries values
// only: a dual plane's tangent is not staged)
__device__ __forceinline__ double sval(double x) { return x; }
__device__ __forceinline__ double sval(float x) { return double(x); }
template <class T>
__device__ __forceinline__ double sval(const Dual<T>& x) {
  return double(x.v);
}

// a stored number as a staged one
template <class E, class T>
__device__ __forceinline__ E staged(const T& x) {
  if constexpr (IsDual<E>::value) return E(x);
  else return E(sval(x));
}

// Block-wide staging of (level, column) planes through LDS slots.  Loads
// and stores issue without barriers so that all planes of a stage are in
// flight together; the caller separates the phases with __syncthreads().
// kEveryPass: issue every load pass, also those past the group's end (all
// lanes then load the group's last element and write nothing) -- a check
// form of the staging, selected with sed_wave = 2; results are identical.
template <class E, int CH, bool kEveryPass = false>
struct SedTile {
  E* lds;       // kSedSlots x kSedCols x row
  int c0, ncol, nz;
  int nzs;      // level stride of a scratch column group
  int row;      // LDS row of one column (sed_row<E>(nz))
  size_t sbase; // scratch offset of the group's first element

  __device__ E* slot(int s) const { return lds + s * (kSedCols * row); }
  // element e of this group in a scratch plane: a base that the block shares
  // (scalar registers) and a 32-bit byte offset, so that a load needs no
  // 64-bit address arithmetic per plane
  template <class T>
  __device__ __forceinline__ T& elem(T* plane, int e) const {
    using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return *reinterpret_cast<T*>(reinterpret_cast<B*>(plane + sbase) + unsigned(e) * unsigned(sizeof(T)));
  }
  // One species' planes (the block's column group of each is one contiguous
  // run): masses and numbers pm and raw speeds ph where the point holds the
  // species (pbit of its flags), tendencies pt where they are stored (tbit),
  // elsewhere dm and zeros.  Every global load is issued into registers before
  // the first LDS write, so the stage waits for one memory latency instead of
  // one per plane and pass (a load-convert-write loop per plane waits for each
  // load before its write).
  // The block has 64 * kSedCols threads and nz <= 64 * CH, so CH passes cover
  // the column group; a pass runs only when the group reaches it (a
  // block-uniform test), and its elements past the group's end load the last
  // one (the index is clamped) and are not written.  kAll: every point is
  // stored (dual planes).
  template <bool kAll, class M, class H, int NM, int NH, int NT>
  __device__ void load_species(const unsigned (&pfe)[CH], unsigned pbit, unsigned tbit, const int (&sm)[NM],
                               const M* const (&pm)[NM], const E (&dm)[NM], const int (&sh)[NH],
                               const H* const (&ph)[NH], const int (&st)[NT], const M* const (&pt)[NT]) const {
    M vm[CH][NM], vt[CH][NT];
    H vh[CH][NH];
    const int n = kSedCols * nz;
#pragma unroll
    for (int it = 0; it < CH; ++it) {
      if (!kEveryPass && it * 64 * kSedCols >= n) break;
      const int e = min(int(threadIdx.x) + it * 64 * kSedCols, n - 1);
      if (kAll || (pfe[it] & pbit)) {
#pragma unroll
        for (int p = 0; p < NM; ++p) vm[it][p] = elem(pm[p], e);
#pragma unroll
        for (int p = 0; p < NH; ++p) vh[it][p] = elem(ph[p], e);
      }
      if (kAll || (pfe[it] & tbit)) {
#pragma unroll
        for (int p = 0; p < NT; ++p) vt[it][p] = elem(pt[p], e);
      }
    }
#pragma unroll
    for (int it = 0; it < CH; ++it) {
      const int e = int(threadIdx.x) + it * 64 * kSedCols;
      if (e < n) {
        const int cc = e % kSedCols, k = e / kSedCols, x = cc * row + k;
        const bool p_ = kAll || (pfe[it] & pbit), t_ = kAll || (pfe[it] & tbit);
#pragma unroll
        for (int p = 0; p < NM; ++p) slot(sm[p])[x] = p_ ? staged<E>(vm[it][p]) : dm[p];
#pragma unroll
        for (int p = 0; p < NH; ++p) slot(sh[p])[x] = p_ ? staged<E>(vh[it][p]) : E(0);
#pragma unroll
        for (int p = 0; p < NT; ++p) slot(st[p])[x] = t_ ? staged<E>(vt[it][p]) : E(0);
      }
    }
  }
  // the first stage in the same way: per-point flags (slot 0, and pfe for this
  // thread's elements), layer depths from the state (slot 1), density (slot 2)
  template <class R, class H>
  __device__ void load_head(const StepArgs<R>& a, const unsigned* pf, const H* rho, unsigned (&pfe)[CH]) const {
    R vz[CH];
    H vh[CH];
    const int n = kSedCols * nz;
#pragma unroll
    for (int it = 0; it < CH; ++it) {
      pfe[it] = 0u;
      if (!kEveryPass && it * 64 * kSedCols >= n) continue;
      const int e = min(int(threadIdx.x) + it * 64 * kSedCols, n - 1);
      const int cc = e % kSedCols, k = e / kSedCols, c = min(c0 + cc, ncol - 1);
      pfe[it] = elem(pf, e) & ~kFlagsChanged;
      vh[it] = elem(rho, e);
      vz[it] = a.f[F_DZ][TEMPO_IDX_STATE(a, c, k)];
    }
#pragma unroll
    for (int it = 0; it < CH; ++it) {
      const int e = int(threadIdx.x) + it * 64 * kSedCols;
      if (e < n) {
        const int cc = e % kSedCols, k = e / kSedCols, x = cc * row + k;
        slot(0)[x] = E(double(pfe[it]));
        slot(1)[x] = c0 + cc < ncol ? staged<E>(vz[it]) : E(0);
        slot(2)[x] = staged<E>(vh[it]);
      }
    }
  }
  // a species' tendencies back to their planes: the sectors (8 consecutive
  // threads: the columns of one level) where one is non-zero or was stored;
  // the flags of the elements that are non-zero gain tbit.  cond: which of
  // the tendencies make an element count (a bit per plane).
  template <bool kAll, class T, int NT>
  __device__ void store_species(unsigned (&pfe)[CH], unsigned tbit, const int (&st)[NT], T* const (&pt)[NT],
                                unsigned cond) const {
#pragma unroll
    for (int it = 0; it < CH; ++it) {
      if (it * 64 * kSedCols >= kSedCols * nz) break;
      const int e = int(threadIdx.x) + it * 64 * kSedCols;
      const int cc = e % kSedCols, k = e / kSedCols;
      const bool in = e < kSedCols * nz && c0 + cc < ncol;
      E v[NT];
      bool counts = false;
#pragma unroll
      for (int p = 0; p < NT; ++p) {
        v[p] = in ? slot(st[p])[cc * row + k] : E(0);
        counts = counts || (((cond >> p) & 1u) && v[p] != E(0));
      }
      if (in && counts && !(pfe[it] & tbit)) pfe[it] |= tbit | kFlagsChanged;
      const bool sector = kAll || ((__ballot(in && (pfe[it] & tbit)) >> (threadIdx.x & 56u)) & 0xffull) != 0ull;
      if (in && sector) {
#pragma unroll
        for (int p = 0; p < NT; ++p) elem(pt[p], e) = T(v[p]);
      }
    }
  }
  // this wavefront's column <-> registers
  template <class T>
  __device__ void get(int s, int w, T (&x)[CH]) const {
    const E* d = slot(s);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + wv::lane();
      x[j] = (k < nz) ? T(d[w * row + k]) : T(0);
    }
  }
  template <class T>
  __device__ void put(int s, int w, const T (&x)[CH]) const {
    E* d = slot(s);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + wv::lane();
      if (k < nz) d[w * row + k] = E(x[j]);
    }
  }
};

// Per-column level geometry held by every lane.
template <int CH, class X = double>
struct SedCol {
  int nzc;                          // active levels
  X odz[CH], orho[CH];
};

// top-down fill (:1768-1789): out(k) = raw(k') at the lowest k' >= k whose
// mass exceeds r1 (0 when none); CFL substeps and ktop from the filled
// speeds in the working precision.  Returns the chunks up to the highest mass:
// above it the speeds are zero and nothing moves, so that neither this nor
// wave_sediment does the chunks above (sedimentation of 25,000 x 90 in FP64
// 214 -> 169 us, of 100,000 x 90 in FP32, bound by its staging, 420 -> 405)
template <class R, int CH, class X>
__device__ __forceinline__ int wave_fill(const X (&mass)[CH], const R (&raw1)[CH],
                                         const R (&raw2)[CH], bool two, bool use_max,
                                         const R (&dz)[CH], int nzc, double dt, X (&out1)[CH],
                                         X (&out2)[CH], int& substeps, int& ktop) {
#pragma clang fp contract(off)  // as the lane-per-column kernel: every operation rounded on its own
  unsigned long long m[CH];
  int chunks = 0;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + wv::lane();
    m[j] = __ballot(k < nzc && mass[j] > kR1);
    if (m[j]) chunks = j + 1;
  }
  int st = 1, kt = 1;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    out1[j] = out2[j] = X(0.0);
    if (CH > 1 && j >= chunks) continue;
    const int l = wv::lane(), k = j * 64 + l;
    int src = -1;
    const unsigned long long mm = m[j] & (~0ull << l);
    if (mm) {
      src = j * 64 + __ffsll((long long)mm) - 1;
    } else {
#pragma unroll
      for (int j2 = j + 1; j2 < CH; ++j2)
        if (src < 0 && m[j2]) src = j2 * 64 + __ffsll((long long)m[j2]) - 1;
    }
    const R r1 = wv::at_level(raw1, src < 0 ? 0 : src);
    const R r2 = two ? wv::at_level(raw2, src < 0 ? 0 : src) : R(0);
    const X v1 = src < 0 ? X(0.0) : X(r1);
    const X v2 = src < 0 ? X(0.0) : X(r2);
    out1[j] = v1;
    out2[j] = v2;
    if (k < nzc) {
      const R vr1 = R(v1), vr2 = R(v2);
      const R vmax = use_max ? mx(vr1, vr2) : vr1;
      if (vmax > R(1.e-3)) {
        kt = max(kt, k + 1);
        const R dz_by_vt = dz[j] / vmax;
        st = max(st, int(R(dt) / dz_by_vt + R(1.0)));
      }
    }
  }
  substeps = wv::imax(st);
  ktop = wv::imax(kt);
  if (ktop == nzc) ktop = nzc - 1;
  return chunks;
}

// one flux-form substep of one field (:1516-1559) in the chunks up to the
// highest non-zero speed (at the top level above it, which the reference
// always updates, the flux is zero, and only a mass below the limit changes);
// returns the surface precipitation increment (0 when the caller does not
// accumulate it)
template <int CH, class X>
__device__ __forceinline__ X wave_sediment(const SedCol<CH, X>& g, X (&xr)[CH], const X (&vt)[CH], X (&xten)[CH],
                                           double limit, int steps, int ktop, int chunks, double dt, bool precip) {
#pragma clang fp contract(off)  // as the lane-per-column kernel: every operation rounded on its own
  const double ost = 1.0 / double(steps);
  X sed[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) sed[j] = j == 0 || j < chunks ? vt[j] * xr[j] : X(0.0);
  const X s0 = wv::read_lane(sed[0], 0);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    if (j > 0 && j >= chunks) continue;
    const X up = wv::above(sed, j);
    const int k = j * 64 + wv::lane();
    if (k < g.nzc && (k == g.nzc - 1 || k <= ktop - 1)) {
      const X flux = (k == g.nzc - 1) ? -sed[j] : (up - sed[j]);
      xten[j] = xten[j] + flux * g.odz[j] * ost * g.orho[j];
      const X v = xr[j] + flux * g.odz[j] * dt * ost;
      xr[j] = v > limit ? v : X(limit);
    }
  }
  if (!precip) return X(0.0);
  const X x0 = wv::read_lane(xr[0], 0);
  return x0 > kLowLimitPrecip ? s0 * dt * ost : X(0.0);
}

// ---- semi-Lagrangian sedimentation on the wavefront --------------------
// semi_sediment (tempo_kernels.hpp) recast with levels across lanes.  What is
// serial there and how it runs here, with the same roundings:
//   heights: summed in level order once per column (they depend on the layer
//     depths alone);
//   the top-down limit of the interface speeds: w(k) is a function of its own
//     unlimited value and of w(k+1), so all levels are updated together from
//     the level above until no level changes (after n rounds the top n levels
//     are final; the chains are short);
//   source cells kb, kt: the limit leaves every departure cell at least 95 %
//     of its layer, so the departure points increase with height and each
//     level finds its cells by bisection instead of following the level below;
//   the surface flux and the decision hash: in level order, on values that
//     every lane reads.
// Arrays that are read at other levels live in LDS rows of the column (kSemiRows
// of nz + 2 doubles): a column's work needs about 30 loads from them per
// level, which in global memory, one lane per column, took 2.43 ms for
// 10,007 columns of 59 levels (157 wavefronts on 256 CUs); here 0.25 ms.
constexpr int kSemiLevels = 128;  // the tile's and these rows' LDS: 119 KB in FP64 at 128 levels
enum SemiRow { SW_ZI, SW_ZA, SW_DZA, SW_QA, SW_QMI, SW_QPI, kSemiRows };
__host__ __device__ constexpr int semi_row(int nz) { return nz + 2; }
__host__ __device__ constexpr size_t semi_lds_bytes(int nz) {
  return size_t(kSedCols) * kSemiRows * semi_row(nz) * sizeof(double);
}

template <int CH>
struct SemiCol {
  double* row;  // this column's LDS rows
  int len;      // semi_row(nz)
  int nz;       // active levels
  double dt;
  double dz[CH], orho[CH];
  __device__ __forceinline__ double& at(int q, int k) const { return row[q * len + k]; }
  // the wavefront's LDS writes before its later reads
  static __device__ __forceinline__ void settle() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  // layer interfaces, summed upwards in level order (every lane the same sum)
  __device__ __forceinline__ void heights() const {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + wv::lane();
      if (k < nz) at(SW_ZA, k) = dz[j];
    }
    settle();
    double z = 0.0;
    at(SW_ZI, 0) = z;
    for (int k = 0; k < nz; ++k) {
      z = z + at(SW_ZA, k);
      at(SW_ZI, k + 1) = z;
    }
    settle();
  }
};

// value of x at level k + 1, k - 1, k - 2 of every lane's level k (0 outside)
template <int CH>
__device__ __forceinline__ double wave_up(const double (&x)[CH], int j) { return wv::above(x, j); }
template <int CH>
__device__ __forceinline__ double wave_down(const double (&x)[CH], int j, int d) {
  // one level at a time: whole-wavefront shift, lane l takes lane l - 1
  double v = wv::dpp<0x138>(j > 0 ? wv::read_lane(x[j > 0 ? j - 1 : 0], 63) : 0.0, x[j]);
  if (d == 2) v = wv::dpp<0x138>(j > 0 ? wv::read_lane(x[j > 0 ? j - 1 : 0], 62) : 0.0, v);
  return v;
}

// one substep of one field (semi_sediment), xr, vt, xten in registers; hash:
// the column's decisions, folded in level order
template <int CH>
__device__ __forceinline__ void wave_semi_sediment(const SemiCol<CH>& g, double (&xr)[CH], double (&xten)[CH],
                                                   const double (&vt)[CH], int steps, double limit, double* precip,
                                                   unsigned& hash) {
#pragma clang fp contract(off)  // as semi_sediment: every operation rounded on its own
  const int nz = g.nz;
  const double dt = g.dt, odt = 1.0 / dt, ost = 1.0 / double(steps), nst = double(steps), con1 = 0.05;
  const double fa1 = 9.0 / 16.0, fa2 = 1.0 / 16.0;
  // interface speeds; level nz has none above it: 0
  double w[CH], w0[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + wv::lane();
    // (every lane takes part in the shuffles; the speeds are 0 above the column)
    const double v = vt[j], up = wave_up(vt, j), dn = wave_down(vt, j, 1), dn2 = wave_down(vt, j, 2);
    double x = 0.0;
    if (k == 0)
      x = v;
    else if (k == 1 || k == nz - 1)
      x = 0.5 * (v + dn);
    else if (k < nz - 1)
      x = fa1 * (v + dn) - fa2 * (up + dn2);
    if (k >= 1 && k < nz && v == 0.0) x = dn;
    w0[j] = w[j] = k < nz ? x : 0.0;
  }
  for (int round = 0; round < nz; ++round) {
    bool moved = false;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + wv::lane();
      const double up = wave_up(w, j);  // 0 at the top interface, the initial value of level nz
      const double decfl = (up - w0[j]) * dt * ost / g.dz[j];
      const double x = k < nz && decfl > con1 ? up - con1 * g.dz[j] * odt * nst : w0[j];
      moved = moved || !(x == w[j]);
      w[j] = x;
    }
    if (!__any(moved)) break;
  }
  // departure points, cells and their contents
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + wv::lane();
    if (k <= nz) g.at(SW_ZA, k) = g.at(SW_ZI, k) - w[j] * dt * ost;
    if (k == 0) g.at(SW_ZA, nz + 1) = g.at(SW_ZI, nz);
  }
  if (nz == 64 * CH && wv::lane() == 0) g.at(SW_ZA, nz) = g.at(SW_ZI, nz) - 0.0 * dt * ost;
  SemiCol<CH>::settle();
  double qa[CH], dza[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + wv::lane();
    if (k < nz) {
      dza[j] = g.at(SW_ZA, k + 1) - g.at(SW_ZA, k);
      qa[j] = xr[j] * g.dz[j] / dza[j];
      g.at(SW_DZA, k) = dza[j];
      g.at(SW_QA, k) = qa[j];
    } else {
      dza[j] = qa[j] = 0.0;
    }
  }
  if (wv::lane() == 0) {
    g.at(SW_DZA, nz) = g.at(SW_ZA, nz + 1) - g.at(SW_ZA, nz);
    g.at(SW_QA, nz) = 0.0;
    g.at(SW_QMI, nz) = g.at(SW_QPI, nz) = 0.0;
  }
  SemiCol<CH>::settle();
  // monotone interface values
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + wv::lane();
    if (k >= nz) continue;
    double qp = qa[j], qm = qa[j];
    if (k > 0) {
      const double dip = (g.at(SW_QA, k + 1) - qa[j]) / (g.at(SW_DZA, k + 1) + dza[j]);
      const double dim = (qa[j] - g.at(SW_QA, k - 1)) / (g.at(SW_DZA, k - 1) + dza[j]);
      if (!(dip * dim <= 0.0)) {
        const double a = qa[j] + 0.5 * (dip + dim) * dza[j];
        const double b = 2.0 * qa[j] - a;
        if (!(a > 0.0 || b < 0.0)) {
          qp = a;
          qm = b;
        }
      }
    }
    g.at(SW_QPI, k) = qp;
    g.at(SW_QMI, k) = qm;
  }
  SemiCol<CH>::settle();
  // remap onto the model levels (1-based kb, kt; level k here is k + 1 there)
  const double zatop = g.at(SW_ZA, nz);
  unsigned out[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + wv::lane();
    out[j] = 0u;
    if (k >= nz) continue;
    const double zlo = g.at(SW_ZI, k), zhi = g.at(SW_ZI, k + 1);
    if (zlo >= zatop) continue;
    // kb: the first of za(1..nz) at or above zlo; kt: the first of
    // za(0..nz+1) at or above zhi
    int a = 1, b = nz, c = 0, d = nz + 1;
    while (__any(a < b || c < d)) {
      const int ab = (a + b) >> 1, cd = (c + d) >> 1;
      const double x = g.at(SW_ZA, ab), y = g.at(SW_ZA, cd);
      if (a < b) {
        if (zlo <= x) b = ab;
        else a = ab + 1;
      }
      if (c < d) {
        if (zhi <= y) d = cd;
        else c = cd + 1;
      }
    }
    const int kb = a, kt = c;
    out[j] = (unsigned(kb) << 16) ^ unsigned(kt);
    double x = xr[j];
    if (kt == kb) {
      const double da = g.at(SW_DZA, kb - 1), za = g.at(SW_ZA, kb - 1), qm = g.at(SW_QMI, kb - 1);
      const double tl = (zlo - za) / da, th = (zhi - za) / da;
      const double tl2 = tl * tl, th2 = th * th;
      const double qqd = 0.5 * (g.at(SW_QPI, kb - 1) - qm);
      const double qqh = qqd * th2 + qm * th;
      const double qql = qqd * tl2 + qm * tl;
      x = (qqh - qql) / (th - tl);
    } else if (kt > kb) {
      const double da = g.at(SW_DZA, kb - 1), qm = g.at(SW_QMI, kb - 1);
      const double tl = (zlo - g.at(SW_ZA, kb - 1)) / da;
      const double tl2 = tl * tl;
      double qqd = 0.5 * (g.at(SW_QPI, kb - 1) - qm);
      const double qql = qqd * tl2 + qm * tl;
      const double dql = g.at(SW_QA, kb - 1) - qql;
      double zsum = (1.0 - tl) * da;
      double qsum = dql * da;
      for (int m = kb; m < kt - 1; ++m) {
        zsum = zsum + g.at(SW_DZA, m);
        qsum = qsum + g.at(SW_QA, m) * g.at(SW_DZA, m);
      }
      const double dt_ = g.at(SW_DZA, kt - 1), qt = g.at(SW_QMI, kt - 1);
      const double th = (zhi - g.at(SW_ZA, kt - 1)) / dt_;
      const double th2 = th * th;
      qqd = 0.5 * (g.at(SW_QPI, kt - 1) - qt);
      const double dqh = qqd * th2 + qt * th;
      zsum = zsum + th * dt_;
      qsum = qsum + dqh * dt_;
      x = qsum / zsum;
    }
    x = x > limit ? x : limit;
    xten[j] = xten[j] + (x - xr[j]) * g.orho[j] * odt;
    xr[j] = x;
  }
  // the decisions: every remapped level's cells, then the first level left out
  bool ended = false;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int n = min(64, nz - j * 64);
    for (int l = 0; l < n && !ended; ++l) {
      const unsigned v = unsigned(__builtin_amdgcn_readlane(int(out[j]), l));
      if (v == 0u) {  // kb >= 1: a remapped level's word is not 0
        hash = decision(hash, 0x100u + unsigned(j * 64 + l + 1));
        ended = true;
      } else {
        hash = decision(hash, v);
      }
    }
  }
  // surface flux: the cells that leave the column
  if (!precip) return;
  double p = *precip;
  for (int k = 0; k < nz; ++k) {
    const double z0 = g.at(SW_ZA, k), z1 = g.at(SW_ZA, k + 1);
    if (!(z0 < 0.0)) break;  // the departure points increase with height
    if (z1 <= 0.0) {
      p = p + g.at(SW_QA, k) * g.at(SW_DZA, k);
      hash = decision(hash, 0x200u + unsigned(k));
    } else if (z1 > 0.0) {
      hash = decision(hash, 0x300u + unsigned(k));
      const double th = (0.0 - z0) / g.at(SW_DZA, k);
      const double th2 = th * th;
      const double qqd = 0.5 * (g.at(SW_QPI, k) - g.at(SW_QMI, k));
      const double qqh = qqd * th2 + g.at(SW_QMI, k) * th;
      p = p + qqh * g.at(SW_DZA, k);
      break;
    }
  }
  *precip = p;
}

// top-down fill of refreshed fall speeds: the value of the lowest level at or
// above each whose mass exceeds r1, 0 above the topmost one
template <class R, int CH>
__device__ __forceinline__ void wave_refill(const double (&mass)[CH], int nzc, const R (&raw1)[CH], const R (&raw2)[CH],
                                            double (&out1)[CH], double (&out2)[CH]) {
  unsigned long long m[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) m[j] = __ballot(j * 64 + wv::lane() < nzc && mass[j] > kR1);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    int src = -1;
    const unsigned long long mm = m[j] & (~0ull << wv::lane());
    if (mm) src = j * 64 + __ffsll((long long)mm) - 1;
#pragma unroll
    for (int j2 = j + 1; j2 < CH; ++j2)
      if (src < 0 && m[j2]) src = j2 * 64 + __ffsll((long long)m[j2]) - 1;
    const R r1 = wv::at_level(raw1, src < 0 ? 0 : src), r2 = wv::at_level(raw2, src < 0 ? 0 : src);
    out1[j] = src < 0 ? 0.0 : double(r1);
    out2[j] = src < 0 ? 0.0 : double(r2);
  }
}

// a level's part of semi_rain_refresh: the checks on the 1-d state with the
// tendencies so far, and the raw fall speeds
template <class R>
__device__ __forceinline__ void semi_rain_level(const StepArgs<R>& a, R rho, R rhof, R qr, R nr, double& qrten,
                                                double& nrten, double& rr, double& rn, R& v1, R& v2) {
  const ConstView<S_t<R>> C = const_view(a.cst);
  Lvl<R> L;
  L.rho = rho;
  L.qrten = R(qrten);
  L.nrten = R(nrten);
  const R q0 = L.qrten, n0 = L.nrten;
  rain_check(C, L, qr, nr, R(a.dt), R(a.odt));
  if (L.qrten != q0) qrten = double(L.qrten);
  if (L.nrten != n0) nrten = double(L.nrten);
  rr = double(L.rr);
  rn = double(L.nr);
  if (L.rr > R(kR1)) rain_fallspeed(C, rhof, R(1.0) / L.ilamr, v1, v2);
}
// ... and of semi_graupel_refresh
template <class R>
__device__ __forceinline__ void semi_graupel_level(const StepArgs<R>& a, R rho, R rhof, R visco, R qg, R ng, R qb,
                                                   double& qgten, double& ngten, double& qbten, double& rg, double& rn,
                                                   double& rb, R& v1, R& v2) {
  const ConstView<S_t<R>> C = const_view(a.cst);
  const bool has_ngqb = a.f[F_NG] && a.f[F_QB];
  Lvl<R> L;
  L.rho = rho;
  L.qgten = R(qgten);
  L.ngten = R(ngten);
  L.qbten = R(qbten);
  const R g0 = L.qgten, n0 = L.ngten, b0 = L.qbten;
  graupel_check(C, L, qg, ng, qb, has_ngqb, R(a.dt), R(a.odt));
  if (L.qgten != g0) qgten = double(L.qgten);
  if (L.ngten != n0) ngten = double(L.ngten);
  if (L.qbten != b0) qbten = double(L.qbten);
  rg = double(L.rg);
  rn = double(L.ng);
  rb = double(L.rb);
  if (L.rg > R(kR1)) graupel_fallspeed(C, L, rhof, visco, a.f[F_QB] != nullptr, v1, v2);
}

// Sedimentation of the column group c0 .. c0 + kSedCols - 1, one wavefront
// per column (64 * kSedCols threads); tile_mem: sed_lds_bytes(nz)
// of LDS.  For a dual working type it runs on the
// values (V, the scalar type) and writes tendencies with zero tangents: the
// tangent-free forward of an adjoint.
// kSemi: semi-Lagrangian rain and graupel, with semi_lds_bytes(nz) more LDS
// behind the tile.
template <class R, int CH = kSedChunks, bool kEveryPass = false, bool kSemi = false, bool kTan = false>
__device__ __forceinline__ void phase_b_group(const StepArgs<R>& a, int c0, void* tile_mem) {
  __shared__ unsigned blk_any;
  const int w = int(threadIdx.x >> 6);
  const int c = c0 + w;
  const bool col_ok = c < a.ncol;
  const size_t plane = a.plane;
  using E = typename SedTypes<R, kTan>::E;
  using X = typename SedTypes<R, kTan>::X;
  const SedTile<E, CH, kEveryPass> T{static_cast<E*>(tile_mem), c0, a.ncol, a.nz, a.nzs, sed_row<E>(a.nz), TEMPO_IDX_SCR(a, c0, 0)};
  const double dt = a.dt;
  Sd_t<R>* sd = a.sd;
  const R* sr = a.sr;
  using V = typename SedTypes<R, kTan>::V;

  SedCol<CH, X> g;
  g.nzc = col_ok ? (a.nlev ? min(max(a.nlev[c], 1), a.nz) : a.nz) : 0;
  if (a.sig && col_ok) {  // signature run: this kernel's decisions are per column (tempo_hip_substeps)
    const size_t n3 = size_t(a.ncol) * size_t(a.nz);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + wv::lane();
      if (k < g.nzc) a.sig[4 * n3 + size_t(k) * a.ncol + c] = a.sig[5 * n3 + size_t(k) * a.ncol + c] = 0u;
    }
  }
  const unsigned cf = col_ok ? a.cf[c] : CF_EXIT;
  const bool live = col_ok && !(cf & CF_EXIT);

  // column flags (which species hold mass) and the level geometry
  constexpr bool kAll = IsDual<R>::value;
  unsigned pfe[CH];  // flags of the elements this thread loads and stores
  if (threadIdx.x == 0) blk_any = 0;
  T.load_head(a, a.pf, sr + SR_RHO * plane, pfe);
  const E r1 = E(S_t<R>(kR1)), r2 = E(S_t<R>(kR2));
  __syncthreads();
  unsigned pfl[CH];
  V dz[CH], rho[CH];
  X rr[CH], vr[CH];
  T.get(0, w, pfl);
  T.get(1, w, dz);
  T.get(2, w, rho);
  unsigned any = 0;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    if (j * 64 + wv::lane() < g.nzc) any |= pfl[j];
    g.odz[j] = X(1.0) / X(dz[j]);
    g.orho[j] = X(1.0) / X(rho[j]);
    vr[j] = X(0.0);
    rr[j] = X(r1);
  }
  any = live ? wv::uor(any) : 0u;
  if (wv::lane() == 0 && any) atomicOr(&blk_any, any);
  __syncthreads();
  const unsigned bany = blk_any;

  // each species' precipitation and substep record wait in LDS for the
  // column's diagnostics
  __shared__ double pr_s[kSedCols][5 * (sizeof(X) / sizeof(double))];
  __shared__ int kst_s[kSedCols][kSubRows];
  X* pr = reinterpret_cast<X*>(pr_s[w]);
  int* kst = kst_s[w];
  if (wv::lane() < 5) pr[wv::lane()] = X(0.0);
  if (wv::lane() < kSubRows) kst[wv::lane()] = wv::lane() < 10 ? 1 : 0;
  auto record = [&](int q, X precip, int steps, int ktop) {
    if (wv::lane() == 0) {
      pr[q] = precip;
      kst[2 * q] = steps;
      kst[2 * q + 1] = ktop;
    }
  };
  SemiCol<CH> sg;
  unsigned hash = 0u;
  V rhof[CH], visco[CH];
  if constexpr (kSemi) {
    double* rows = reinterpret_cast<double*>(static_cast<char*>(tile_mem) + sed_lds_bytes<E>(a.nz));
    sg.row = rows + w * (kSemiRows * semi_row(a.nz));
    sg.len = semi_row(a.nz);
    sg.nz = g.nzc;
    sg.dt = dt;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + wv::lane();
      sg.dz[j] = double(dz[j]);
      sg.orho[j] = g.orho[j];
      rhof[j] = visco[j] = V(0);
      if ((any & (PF_QR | PF_QG)) && k < g.nzc) {
        rhof[j] = value(sr[SR_RHOF * plane + TEMPO_IDX_SCR(a, c, k)]);
        visco[j] = value(sr[SR_VISCO * plane + TEMPO_IDX_SCR(a, c, k)]);
      }
    }
    if (any & (PF_QR | PF_QG)) sg.heights();
  }

  // ---- rain (:603-630) ----
  if (bany & PF_QR) {
    X xn[CH], tr[CH], tn[CH], v2[CH];
    V raw1[CH], raw2[CH];
    T.template load_species<kAll>(pfe, PF_QR, PF_TR, {3, 0}, {sd + SD_RR * plane, sd + SD_NR * plane}, {r1, r2}, {4, 5},
                                  {sr + SR_VTRR * plane, sr + SR_VTNR * plane}, {1, 2},
                                  {sd + SD_QRTEN * plane, sd + SD_NRTEN * plane});
    __syncthreads();
    T.get(3, w, rr);
    T.get(0, w, xn);
    T.get(1, w, tr);
    T.get(2, w, tn);
    T.get(4, w, raw1);
    T.get(5, w, raw2);
    if (any & PF_QR) {
      int steps, ktop;
      X pq = X(0.0);
      const int ch = wave_fill(rr, raw1, raw2, true, true, dz, g.nzc, dt, vr, v2, steps, ktop);
      if constexpr (kSemi) {  // (:599-615): far fewer substeps, fall speeds refreshed after each
        steps = max(int(R(steps) / R(10.0)) + 1, 1);
        V q[CH], qn[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
          const int k = j * 64 + wv::lane();
          const bool in = k < g.nzc;
          q[j] = in ? a.fa[F_QR][TEMPO_IDX_STATE(a, c, k)] : V(0);
          qn[j] = in ? a.fa[F_NR][TEMPO_IDX_STATE(a, c, k)] : V(0);
        }
        for (int n = 0; n < steps; ++n) {
          wave_semi_sediment(sg, rr, tr, vr, steps, kR1, &pq, hash);
          wave_semi_sediment(sg, xn, tn, v2, steps, kR2, nullptr, hash);
#pragma unroll
          for (int j = 0; j < CH; ++j) {
            raw1[j] = raw2[j] = V(0);
            if (j * 64 + wv::lane() < g.nzc)
              semi_rain_level(a, rho[j], rhof[j], q[j], qn[j], tr[j], tn[j], rr[j], xn[j], raw1[j], raw2[j]);
          }
          wave_refill(rr, g.nzc, raw1, raw2, vr, v2);
        }
      } else for (int n = 0; n < steps; ++n) {
        pq += wave_sediment(g, rr, vr, tr, kR1, steps, ktop, ch, dt, true);
        wave_sediment(g, xn, v2, tn, kR2, steps, ktop, ch, dt, false);
      }
      record(0, pq, steps, ktop);
      if (kSemi && wv::lane() == 0) kst[10] = int(hash);
    }
    T.put(1, w, tr);
    T.put(2, w, tn);
    __syncthreads();
    T.template store_species<kAll>(pfe, PF_TR, {1, 2}, {sd + SD_QRTEN * plane, sd + SD_NRTEN * plane}, 3u);
    __syncthreads();
  }

  // ---- graupel (:632-660) ----
  if (bany & PF_QG) {
    X xg[CH], xn[CH], xb[CH], tg[CH], tn[CH], tb[CH];
    X v1[CH], v2[CH];
    V raw1[CH], raw2[CH];
    const E rb0 = E(S_t<R>(kM3ToL) * S_t<R>(kR1) / rho_g<S_t<R>>(kIdxBg1));
    T.template load_species<kAll>(pfe, PF_QG, PF_TG, {0, 1, 2}, {sd + SD_RG * plane, sd + SD_NG * plane, sd + SD_RB * plane},
                                  {r1, r2, rb0}, {7, 3}, {sr + SR_VTRG * plane, sr + SR_VTNG * plane}, {4, 5, 6},
                                  {sd + SD_QGTEN * plane, sd + SD_NGTEN * plane, sd + SD_QBTEN * plane});
    __syncthreads();
    T.get(0, w, xg);
    T.get(1, w, xn);
    T.get(2, w, xb);
    T.get(4, w, tg);
    T.get(5, w, tn);
    T.get(6, w, tb);
    T.get(7, w, raw1);
    T.get(3, w, raw2);
    if (any & PF_QG) {
      int steps, ktop;
      X pq = X(0.0);
      hash = 0u;
      const int ch = wave_fill(xg, raw1, raw2, true, false, dz, g.nzc, dt, v1, v2, steps, ktop);
      const double rb_lim = kM3ToL * kR1 / 800.0;
      if constexpr (kSemi) {  // (:641-667)
        steps = max(int(R(steps) / R(10.0)) + 1, 1);
        const bool has_ngqb = a.f[F_NG] && a.f[F_QB];
        V q[CH], qn[CH], qb[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
          const int k = j * 64 + wv::lane();
          const bool in = k < g.nzc;
          q[j] = in ? a.fa[F_QG][TEMPO_IDX_STATE(a, c, k)] : V(0);
          qn[j] = in && has_ngqb ? a.fa[F_NG][TEMPO_IDX_STATE(a, c, k)] : V(0);
          qb[j] = in && has_ngqb ? a.fa[F_QB][TEMPO_IDX_STATE(a, c, k)] : V(0);
        }
        for (int n = 0; n < steps; ++n) {
          wave_semi_sediment(sg, xg, tg, v1, steps, kR1, &pq, hash);
          wave_semi_sediment(sg, xn, tn, v2, steps, kR2, nullptr, hash);
          wave_semi_sediment(sg, xb, tb, v1, steps, rb_lim, nullptr, hash);
#pragma unroll
          for (int j = 0; j < CH; ++j) {
            raw1[j] = raw2[j] = V(0);
            if (j * 64 + wv::lane() < g.nzc)
              semi_graupel_level(a, rho[j], rhof[j], visco[j], q[j], qn[j], qb[j], tg[j], tn[j], tb[j], xg[j], xn[j],
                                 xb[j], raw1[j], raw2[j]);
          }
          wave_refill(xg, g.nzc, raw1, raw2, v1, v2);
        }
      } else for (int n = 0; n < steps; ++n) {
        pq += wave_sediment(g, xg, v1, tg, kR1, steps, ktop, ch, dt, true);
        wave_sediment(g, xn, v2, tn, kR2, steps, ktop, ch, dt, false);
        wave_sediment(g, xb, v1, tb, rb_lim, steps, ktop, ch, dt, false);
      }
      record(1, pq, steps, ktop);
      if (kSemi && wv::lane() == 0) kst[11] = int(hash);
    }
    T.put(4, w, tg);
    T.put(5, w, tn);
    T.put(6, w, tb);
    __syncthreads();
    T.template store_species<kAll>(pfe, PF_TG, {4, 5, 6},
                                   {sd + SD_QGTEN * plane, sd + SD_NGTEN * plane, sd + SD_QBTEN * plane}, 7u);
    __syncthreads();
  }

  // ---- snow (:662-697): mixes in the filled rain speed where snow melts,
  // with the rain mass after rain sedimentation ----
  if (bany & PF_QS) {
    X xs[CH], ts[CH], v1[CH];
    V raw[CH];
    T.template load_species<kAll>(pfe, PF_QS, PF_TS, {0}, {sd + SD_RS * plane}, {r1}, {2}, {sr + SR_VTS * plane}, {1},
                                  {sd + SD_QSTEN * plane});
    __syncthreads();
    T.get(0, w, xs);
    T.get(1, w, ts);
    T.get(2, w, raw);
    if (any & PF_QS) {
#pragma clang fp contract(off)  // the snow-rain speed mix, as the lane-per-column kernel
      V vraw[CH];
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        V v = raw[j];
        if (pfl[j] & PF_SNOWMIX) {
          // the top level, which rain's sedimentation always updates, holds at
          // least r1, also in a chunk above the highest mass, left out there
          if (CH > 1 && !kSemi && (any & PF_QR) && j * 64 + wv::lane() == g.nzc - 1 && !(rr[j] > kR1)) rr[j] = X(kR1);
          const V sr_ = V(xs[j] / (xs[j] + rr[j]));
          v = v * sr_ + (V(1.0) - sr_) * V(vr[j]);
        }
        vraw[j] = v;
      }
      X unused[CH];
      int steps, ktop;
      const int ch = wave_fill(xs, vraw, vraw, false, false, dz, g.nzc, dt, v1, unused, steps, ktop);
      X pq = X(0.0);
      for (int n = 0; n < steps; ++n) pq += wave_sediment(g, xs, v1, ts, kR1, steps, ktop, ch, dt, true);
      record(2, pq, steps, ktop);
    }
    T.put(1, w, ts);
    __syncthreads();
    T.template store_species<kAll>(pfe, PF_TS, {1}, {sd + SD_QSTEN * plane}, 1u);
    __syncthreads();
  }

  // ---- ice (:699-715): one call with steps = substeps ----
  if (bany & PF_QI) {
    X xi[CH], xn[CH], ti[CH], tn[CH], v1[CH], v2[CH];
    V raw1[CH], raw2[CH];
    T.template load_species<kAll>(pfe, PF_QI, PF_TI, {0, 1}, {sd + SD_RI * plane, sd + SD_NI * plane}, {r1, r2}, {5, 6},
                                  {sr + SR_VTRI * plane, sr + SR_VTNI * plane}, {2, 4},
                                  {sd + SD_QITEN * plane, sd + SD_NITEN * plane});
    __syncthreads();
    T.get(0, w, xi);
    T.get(1, w, xn);
    T.get(2, w, ti);
    T.get(4, w, tn);
    T.get(5, w, raw1);
    T.get(6, w, raw2);
    if (any & PF_QI) {
      int steps, ktop;
      const int ch = wave_fill(xi, raw1, raw2, true, false, dz, g.nzc, dt, v1, v2, steps, ktop);
      const X pq = wave_sediment(g, xi, v1, ti, kR1, steps, ktop, ch, dt, true);
      wave_sediment(g, xn, v2, tn, kR2, steps, ktop, ch, dt, false);
      record(3, pq, steps, ktop);
    }
    T.put(2, w, ti);
    T.put(4, w, tn);
    __syncthreads();
    T.template store_species<kAll>(pfe, PF_TI, {2, 4}, {sd + SD_QITEN * plane, sd + SD_NITEN * plane}, 3u);
    __syncthreads();
  }

  // ---- cloud (:717-727, cloud_fallspeed :1945-1977): below 500 m only ----
  if (bany & PF_QC) {
    X xc[CH], xn[CH], tc[CH], tn[CH], v1[CH], v2[CH];
    V raw1[CH], raw2[CH];
    const bool has_nc = a.f[F_NC] != nullptr;
    T.template load_species<kAll>(pfe, PF_QC, PF_TC, {0, 1}, {sd + SD_RC * plane, sd + SD_NC * plane},
                                  {r1, E(S_t<R>(kNtCMin))}, {5, 6}, {sr + SR_VTRC * plane, sr + SR_VTNC * plane}, {2, 4},
                                  {sd + SD_QCTEN * plane, sd + SD_NCTEN * plane});
    __syncthreads();
    T.get(0, w, xc);
    T.get(1, w, xn);
    T.get(2, w, tc);
    T.get(4, w, tn);
    T.get(5, w, raw1);
    T.get(6, w, raw2);
    if (any & PF_QC) {
      int kt = 1;
      V hgt = V(0.0);
      for (int k = 0; k < g.nzc - 1; ++k) {  // uniform loop: every lane follows level k
        if (wv::at_uniform(xc, k) > kR2) kt = k + 1;
        hgt = hgt + wv::at_uniform(dz, k);
        if (hgt > V(500.0)) break;
      }
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int k = j * 64 + wv::lane();
        v1[j] = (k < kt) ? X(raw1[j]) : X(0.0);
        v2[j] = (k < kt) ? X(raw2[j]) : X(0.0);
      }
      // cloud settles into levels without any: theirs is a number tendency too
      if constexpr (!kAll) {
        if (!has_nc) {
#pragma unroll
          for (int j = 0; j < CH; ++j) {
            const bool fed = wv::above(v1, j) != X(0.0);
            const int k = j * 64 + wv::lane();
            if (fed && k < kt && !(a.pf[TEMPO_IDX_SCR(a, c, k)] & PF_TC)) tn[j] = X(sd[SD_NCTEN * plane + TEMPO_IDX_SCR(a, c, k)]);
          }
        }
      }
      const X pq = wave_sediment(g, xc, v1, tc, kR1, 1, kt, (kt + 63) / 64, dt, true);
      wave_sediment(g, xn, v2, tn, kR2, 1, kt, (kt + 63) / 64, dt, false);
      record(4, pq, 1, kt);
    }
    T.put(2, w, tc);
    T.put(4, w, tn);
    __syncthreads();
    T.template store_species<kAll>(pfe, PF_TC, {2, 4}, {sd + SD_QCTEN * plane, sd + SD_NCTEN * plane},
                                   has_nc ? 3u : 1u);
  }
  if (!kAll) {  // the flags the final update reads
#pragma unroll
    for (int it = 0; it < CH; ++it) {
      const int e = int(threadIdx.x) + it * 64 * kSedCols;
      if (e < kSedCols * a.nz && c0 + e % kSedCols < a.ncol && (pfe[it] & kFlagsChanged))
        T.elem(a.pf, e) = pfe[it] & ~kFlagsChanged;
    }
  }

  if (!col_ok || wv::lane() != 0) return;
  for (int q = 0; q < 5; ++q) a.precip[size_t(q) * a.ncol + c] = pr[q];
  if (a.ksub)
    for (int q = 0; q < kSubRows; ++q) a.ksub[size_t(q) * a.ncol + c] = kst[q];
  // column diagnostics (src/module_mp_tempo_main.F90:784-794, driver :452-457)
  const size_t d2 = size_t(c % a.ni) + size_t(c / a.ni) * a.d2ldj;
  const R rain = R(pr[0]), graupel = R(pr[1]), snow = R(pr[2]), ice = R(pr[3]), cloud = R(pr[4]);
  if (a.d2[D2_RAIN]) a.d2[D2_RAIN][d2] = rain;
  if (a.d2[D2_ICE]) a.d2[D2_ICE][d2] = ice;
  if (a.d2[D2_SNOW]) a.d2[D2_SNOW][d2] = snow;
  if (a.d2[D2_GRAUPEL]) a.d2[D2_GRAUPEL][d2] = graupel;
  if (a.d2[D2_FROZEN])
    a.d2[D2_FROZEN][d2] = live ? (ice + snow + graupel) / (ice + snow + graupel + rain + R(kR1)) : R(0);
  if (a.d2[D2_FRZRAIN]) {
    R frz = R(0);
    if (live && (sr[SR_TEMP * plane + TEMPO_IDX_SCR(a, c, 0)] - R(kT0)) < R(-0.5)) frz = rain + cloud;
    a.d2[D2_FRZRAIN][d2] = frz;
  }
  if (a.d2[D2_HAIL_SFC]) a.d2[D2_HAIL_SFC][d2] = R(0);
  if (a.d2[D2_HAIL_COL]) a.d2[D2_HAIL_COL][d2] = R(0);
}

// Waves per SIMD by chunks, as many as the registers allow next to no spills:
// one chunk is held to 7 (50 VGPRs in FP32, none spilled, where 8 run), two to 6
// (80 VGPRs, 20 B spilled), three and four take what they need (110, 138).  A
// spill is a scratch-memory access in every stage and dominates soon: two
// chunks held to 8 waves (128 B of spills) took 1.20 ms at 100,000 x 90 against
// 0.50 at 6 (52 B then) and 0.49 at 5; now 0.40 at 6.
// Against one lane per column the wavefront form takes, for the whole step,
// 0.33 instead of 2.93 ms at 8,191 x 160 (FP32; one lane per column is 128
// wavefronts on 256 CUs).
constexpr int sed_waves(int chunks) { return chunks <= 1 ? 7 : chunks == 2 ? 6 : chunks == 3 ? 4 : 3; }
template <class R, int CH, bool kEveryPass = false>
__global__ void __launch_bounds__(64 * kSedCols) __attribute__((amdgpu_waves_per_eu(sed_waves(CH)))) k_phase_b_wave(StepArgs<R> a) {
  extern __shared__ double tile_mem[];  // sed_lds_bytes<SedStage<R>>(nz)
  phase_b_group<R, CH, kEveryPass>(a, int(blockIdx.x) * kSedCols, tile_mem);
}

// ... with semi-Lagrangian rain and graupel
template <class R, int CH>
__global__ void __launch_bounds__(64 * kSedCols) k_phase_b_semi_wave(StepArgs<R> a) {
  extern __shared__ double tile_mem[];  // sed_lds_bytes<SedStage<R>>(nz) + semi_lds_bytes(nz)
  phase_b_group<R, CH, false, true>(a, int(blockIdx.x) * kSedCols, tile_mem);
}
template <class R>
void launch_phase_b_semi_wave(const StepArgs<R>& a, hipStream_t s) {
  const dim3 g(unsigned((a.ncol + kSedCols - 1) / kSedCols)), b(64 * kSedCols);
  const size_t lds = sed_lds_bytes<SedStage<R>>(a.nz) + semi_lds_bytes(a.nz);
  if (a.nz <= 64)
    hipLaunchKernelGGL((k_phase_b_semi_wave<R, 1>), g, b, lds, s, a);
  else
    hipLaunchKernelGGL((k_phase_b_semi_wave<R, 2>), g, b, lds, s, a);
}

// ... of the tangent-linear step: duals throughout
template <class R, int CH>
__global__ void __launch_bounds__(64 * kSedCols) k_phase_b_tan_wave(StepArgs<R> a) {
  extern __shared__ double tile_mem[];  // sed_lds_bytes<W_t<R>>(nz)
  phase_b_group<R, CH, false, false, true>(a, int(blockIdx.x) * kSedCols, tile_mem);
}
// the four launches of one tangent-linear step; sedimentation one wavefront
// per column in flux form up to kSedLevels levels, else one lane per column.
// 8,192 columns are 128 wavefronts at one lane per column: 840 of the step's
// 1364 us at 64 levels (FP32), against 63 of 553 us here.
template <class D>
hipError_t launch_step_tlm_impl(const StepArgs<D>& a, const LaunchCfg& lc, Dual<double>* vtbuf, hipStream_t s) {
  launch_prepass(a, s);
  hipLaunchKernelGGL(k_phase_a<D>, level_grid(a, 256), dim3(256), 0, s, a);
  if (lc.sed_wave && a.nz <= kSedLevels && !a.fl.semi_sedi) {
    const dim3 g(unsigned((a.ncol + kSedCols - 1) / kSedCols)), b(64 * kSedCols);
    const size_t lds = sed_lds_bytes<Dual<double>>(a.nz);
    if (a.nz <= 64)
      hipLaunchKernelGGL((k_phase_b_tan_wave<D, 1>), g, b, lds, s, a);
    else
      hipLaunchKernelGGL((k_phase_b_tan_wave<D, 2>), g, b, lds, s, a);
  } else {
    hipLaunchKernelGGL(k_phase_b<D>, dim3(unsigned((a.ncol + 127) / 128)), dim3(128), 0, s, a, vtbuf);
  }
  hipLaunchKernelGGL(k_phase_c<D>, level_grid(a, 256), dim3(256), 0, s, a);
  return hipGetLastError();
}

// nz <= kSedMaxLevels (dual working types: kSedLevels)
template <class R>
void launch_phase_b_wave(const StepArgs<R>& a, hipStream_t s) {
  const dim3 g(unsigned((a.ncol + kSedCols - 1) / kSedCols)), b(64 * kSedCols);
  const size_t lds = sed_lds_bytes<SedStage<R>>(a.nz);
  if (a.nz <= 64)
    hipLaunchKernelGGL((k_phase_b_wave<R, 1>), g, b, lds, s, a);
  else if (a.nz <= 128)
    hipLaunchKernelGGL((k_phase_b_wave<R, 2>), g, b, lds, s, a);
  else if constexpr (!IsDual<R>::value) {
    if (a.nz <= 192)
      hipLaunchKernelGGL((k_phase_b_wave<R, 3>), g, b, lds, s, a);
    else
      hipLaunchKernelGGL((k_phase_b_wave<R, 4>), g, b, lds, s, a);
  }
}

// ------------------------------------------------------------- launch ----
// The four launches of one step.  ga carries the same arguments as a in the
// level-local kernels' working type: a itself, or its Sig<T> view for a run
// that records branch signatures (StepArgs<T> and StepArgs<Sig<T>> have the
// same layout).
template <class T, class RA>
hipError_t launch_step_impl(const StepArgs<T>& args, const StepArgs<RA>& gargs, const LaunchCfg& lc, double* vtbuf,
                            hipStream_t s, hipEvent_t* ev) {
  StepArgs<T> a = args;
  StepArgs<RA> ga = gargs;
  // the lane-per-column kernel reads every point's planes.  The clear-air path
  // leaves out planes that the semi-Lagrangian refresh, the melting level and
  // the network's one-moment cloud number need, is the general path's result
  // only where condensation runs, and is off in signature runs, whose records
  // are of the decisions themselves.
  const bool semi_wave = lc.sed_wave && a.nz <= kSemiLevels && a.fl.semi_sedi && !a.sig;
  const bool wave = semi_wave || (lc.sed_wave && a.nz <= kSedMaxLevels && !a.fl.semi_sedi);
  const bool clear = wave && !a.sig && !a.fl.semi_sedi && !(a.fl.refl_from_melting && a.fl.refl10cm) &&
                     !(a.fl.ml_for_nc && !a.f[F_NC]) && !a.fl.turn_off_micro && a.fl.cloud_condensation;
  a.sparse = ga.sparse = (wave ? SPARSE_PLANES : 0) | (clear ? SPARSE_CLEAR : 0);
  if (ev) (void)hipEventRecord(ev[0], s);
  launch_prepass(a, s);
  if (ev) (void)hipEventRecord(ev[1], s);
  // FP64 with the registers of two waves per SIMD has next to no spills and is
  // faster while the launch is one or two rounds of them at most (2,048 run
  // at once): 1 column x 60 122 -> 115 us, 2,000 x 90 (2,880 wavefronts) 206 ->
  // 186, 3,000 x 90 (4,230) 272 -> 265; 5,000 x 60 (4,740) 265 -> 275, 25,000 x
  // 90 1573 -> 1585.  FP32 gains nothing at any size.
  const bool fewer = lc.waves_a >= 0 ? lc.waves_a == 1
                                     : sizeof(T) == 8 && size_t((a.ncol + 63) / 64) * size_t(a.nz) <= 4096;
  if (fewer && std::is_same<RA, T>::value)
    hipLaunchKernelGGL((k_phase_a<RA, WavesPerEu<RA>::a_alt>), level_grid(a, lc.block_a), dim3(unsigned(lc.block_a)),
                       0, s, ga);
  else
    hipLaunchKernelGGL(k_phase_a<RA>, level_grid(a, lc.block_a), dim3(unsigned(lc.block_a)), 0, s, ga);
  if (ev) (void)hipEventRecord(ev[2], s);
  if (lc.sed_wave == 2 && a.nz <= kSedLevels && !a.fl.semi_sedi)
    hipLaunchKernelGGL((k_phase_b_wave<T, kSedChunks, true>), dim3(unsigned((a.ncol + kSedCols - 1) / kSedCols)),
                       dim3(64 * kSedCols), sed_lds_bytes<SedStage<T>>(a.nz), s, a);
  else if (semi_wave)
    launch_phase_b_semi_wave(a, s);
  else if (wave)
    launch_phase_b_wave(a, s);
  else
    hipLaunchKernelGGL(k_phase_b<T>, dim3(unsigned((a.ncol + 127) / 128)), dim3(128), 0, s, a, vtbuf);
  if (a.fl.refl_from_melting && a.fl.refl10cm && a.d3[D3_REFL]) {
    hipLaunchKernelGGL(k_melt_level<T>, dim3(unsigned((a.ncol + 63) / 64)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_melt_refl<T>, level_grid(a, 256), dim3(256), 0, s, a);
  }
  if (ev) (void)hipEventRecord(ev[3], s);
  hipLaunchKernelGGL(k_phase_c<RA>, level_grid(a, lc.block_c), dim3(unsigned(lc.block_c)), 0, s, ga);
  if (ev) (void)hipEventRecord(ev[4], s);
  return hipGetLastError();
}

template <class T>
StepArgs<Sig<T>> sig_args(const StepArgs<T>& a) {
  static_assert(sizeof(StepArgs<Sig<T>>) == sizeof(StepArgs<T>), "StepArgs layout");
  StepArgs<Sig<T>> g;
  std::memcpy(&g, &a, sizeof(a));
  return g;
}

}  // namespace tempo
