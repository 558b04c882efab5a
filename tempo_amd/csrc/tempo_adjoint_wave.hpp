// S^T with one wavefront per column, levels across lanes (nz <= 128): the
// serial column adjoint of tempo_adjoint.hpp recast on the wavefront
// primitives of the sedimentation kernel.  Every substep's adjoint is a
// two-point stencil in the level index (the flux of level k reads the
// sedimentation rate of k+1), so all levels update at once: the rate
// cotangent of level k collects its own flux cotangent and that of level
// k-1 by a one-lane shift.  Fill sources come from a ballot of the levels
// holding mass; the cotangents of the filled speeds are gathered back to
// their source levels through a per-wavefront LDS row, summed in level
// order.
#pragma once

#include "tempo_adjoint.hpp"
#include "tempo_sedi.hpp"

namespace tempo {

namespace wv {
// value of x at level k-1 for every lane's level k in chunk j (0 below level 0)
template <int CH, class T>
__device__ __forceinline__ T below(const T (&x)[CH], int j) {
  return dpp<0x138>(j > 0 ? read_lane(x[j > 0 ? j - 1 : 0], 63) : T(0), x[j]);
}
}  // namespace wv

template <int CH>
struct WaveCol {
  int nzc, top;
  double dt;
  double odz[CH], orho[CH];
};

// fill sources: lowest level >= k whose mass exceeds r1 (-1: none)
template <int CH>
__device__ __forceinline__ void wave_fill_src(const double (&mass)[CH], int nzc, int (&src)[CH],
                                              unsigned long long (&m)[CH]) {
#pragma unroll
  for (int j = 0; j < CH; ++j) m[j] = __ballot(j * 64 + wv::lane() < nzc && mass[j] > kR1);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int l = wv::lane();
    int s = -1;
    const unsigned long long mm = m[j] & (~0ull << l);
    if (mm) {
      s = j * 64 + __ffsll((long long)mm) - 1;
    } else {
#pragma unroll
      for (int j2 = j + 1; j2 < CH; ++j2)
        if (s < 0 && m[j2]) s = j2 * 64 + __ffsll((long long)m[j2]) - 1;
    }
    src[j] = s;
  }
}

// out(k) = raw(src(k)) or 0
template <int CH>
__device__ __forceinline__ void wave_gather(const double (&raw)[CH], const int (&src)[CH],
                                            double (&out)[CH]) {
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const double r = wv::at_level(raw, src[j] < 0 ? 0 : src[j]);
    out[j] = src[j] < 0 ? 0.0 : r;
  }
}

// acc(k') += sum over levels k with src(k) = k' of vb(k), summed in level order
template <int CH>
__device__ __forceinline__ void wave_scatter(const double (&vb)[CH], const int (&src)[CH],
                                             const unsigned long long (&m)[CH], double* row, int nzc,
                                             double (&acc)[CH]) {
#pragma unroll
  for (int j = 0; j < CH; ++j) row[j * 64 + wv::lane()] = vb[j];
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + wv::lane();
    if (k >= nzc || !((m[j] >> wv::lane()) & 1ull)) continue;
    // previous source level below k (its segment ends there)
    int lo = -1;
    const unsigned long long below_mask = wv::lane() ? (m[j] & ((1ull << wv::lane()) - 1ull)) : 0ull;
    if (below_mask) {
      lo = j * 64 + 63 - __clzll((long long)below_mask);
    } else {
#pragma unroll
      for (int j2 = j - 1; j2 >= 0; --j2)
        if (lo < 0 && m[j2]) lo = j2 * 64 + 63 - __clzll((long long)m[j2]);
    }
    double s = 0.0;
    for (int kk = lo + 1; kk <= k; ++kk) s += row[kk];
    acc[j] += s;
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// one field's substeps backwards (see sed_adjoint in tempo_adjoint.hpp)
template <int CH>
__device__ __forceinline__ void wave_sed_adjoint(const WaveCol<CH>& q, const double (&xr0)[CH],
                                                 const double (&vt)[CH], const double (&tb)[CH],
                                                 double limit, int nsub, int steps, int ktop, double pbar,
                                                 double (&xb)[CH], double (&vb)[CH],
                                                 double (&rhob)[CH]) {
  // every operation rounded on its own, as in the forward sedimentation it
  // recomputes (so that the recomputed masses and clamps are the forward's)
#pragma clang fp contract(off)
  const double ost = 1.0 / double(steps), dt = q.dt;
  auto updated = [&](int k) { return k < q.nzc && (k == q.top || k <= ktop - 1); };
  for (int n = nsub - 1; n >= 0; --n) {
    double xr[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) xr[j] = xr0[j];
    for (int r = 0; r < n; ++r) {
      double sed[CH];
#pragma unroll
      for (int j = 0; j < CH; ++j) sed[j] = vt[j] * xr[j];
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const double up = wv::above(sed, j);
        const int k = j * 64 + wv::lane();
        if (updated(k)) {
          const double flux = (k == q.top) ? -sed[j] : (up - sed[j]);
          const double v = xr[j] + flux * q.odz[j] * dt * ost;
          xr[j] = v > limit ? v : limit;
        }
      }
    }
    double sed[CH], fb[CH], post[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) sed[j] = vt[j] * xr[j];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const double up = wv::above(sed, j);
      const int k = j * 64 + wv::lane();
      fb[j] = 0.0;
      post[j] = xr[j];
      if (updated(k)) {
        const double flux = (k == q.top) ? -sed[j] : (up - sed[j]);
        const double v = xr[j] + flux * q.odz[j] * dt * ost;
        const double vbar = v > limit ? xb[j] : 0.0;
        fb[j] = vbar * q.odz[j] * dt * ost + tb[j] * q.odz[j] * ost * q.orho[j];
        if (tb[j] != 0.0) rhob[j] += -q.orho[j] * q.orho[j] * tb[j] * flux * q.odz[j] * ost;
        xb[j] = vbar;
        post[j] = v > limit ? v : limit;
      }
    }
    const double x0post = wv::read_lane(post[0], 0);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const double fbl = wv::below(fb, j);
      const int k = j * 64 + wv::lane();
      if (k >= q.nzc) continue;
      double sb = updated(k) ? -fb[j] : 0.0;
      if (k >= 1 && updated(k - 1) && k - 1 != q.top) sb += fbl;
      if (k == 0 && pbar != 0.0 && x0post > kLowLimitPrecip) sb += pbar * dt * ost;
      xb[j] += sb * vt[j];
      vb[j] += sb * xr[j];
    }
  }
}

// S^T of kScrW columns, a wavefront each.  A column's levels lie 64 bytes
// apart in every plane, so a wavefront reading its own column touches 64
// lines per access; the block therefore moves whole planes of its column
// group through LDS, consecutive threads on consecutive elements, and a
// wavefront picks its column's row up from there (16,384 x 64 FP32, 30 planes
// read and 20 written: 162 us, 318 with direct accesses).  The planes of a
// species that no column of the block holds are only zeroed.
template <class D, int CH>
__global__ void __launch_bounds__(64 * kScrW) k_adj_sed_wave(StepArgs<D> a, AdjArgs g) {
  // every operation rounded on its own, as in the forward sedimentation it
  // recomputes (so that the recomputed masses and clamps are the forward's)
#pragma clang fp contract(off)
  constexpr int kSlots = 6, kRow = 64 * CH + 8;  // rows 8 doubles apart in the banks
  __shared__ double tile[kSlots][kScrW][kRow];
  __shared__ double rows[kScrW][64 * CH];
  __shared__ unsigned any_w[kScrW];
  using R = D;
  const int w = int(threadIdx.x >> 6), l = wv::lane();
  const int c0 = int(blockIdx.x) * kScrW, c = c0 + w;
  const bool live = c < a.ncol && !(a.cf[c] & CF_EXIT);
  double* row = rows[w];
  const size_t plane = a.plane, base = TEMPO_IDX_SCR(a, c0, 0);
  const int count = a.nz * kScrW;  // the block's elements of a plane, contiguous from base
  WaveCol<CH> q;
  q.nzc = !live ? 0 : a.nlev ? min(max(a.nlev[c], 1), a.nz) : a.nz;
  q.top = q.nzc - 1;
  q.dt = a.dt;
  // block-wide moves between a plane and a slot
  auto stage = [&](int slot, const auto* p) {
    for (int e = int(threadIdx.x); e < count; e += 64 * kScrW) tile[slot][e % kScrW][e / kScrW] = double(value(p[base + e]));
  };
  auto stage_sd = [&](int slot, int f) { stage(slot, a.sd + size_t(f) * plane); };
  auto stage_sr = [&](int slot, int f) { stage(slot, a.sr + size_t(f) * plane); };
  auto stage_ub = [&](int slot, int m) { stage(slot, g.ubar + size_t(m) * plane); };
  auto flush = [&](int slot, int z) {
    double* p = g.zbar + size_t(z) * plane + base;
    for (int e = int(threadIdx.x); e < count; e += 64 * kScrW) p[e] = tile[slot][e % kScrW][e / kScrW];
  };
  auto clear_z = [&](int z) {
    double* p = g.zbar + size_t(z) * plane + base;
    for (int e = int(threadIdx.x); e < count; e += 64 * kScrW) p[e] = 0.0;
  };
  // the wavefront's column of a slot; its row only, so the moves above need
  // the block's barriers and these do not
  auto get = [&](int slot, double (&x)[CH]) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + l;
      x[j] = k < q.nzc ? tile[slot][w][k] : 0.0;
    }
  };
  auto put = [&](int slot, const double (&x)[CH]) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + l;
      tile[slot][w][k] = k < q.nzc ? 0.0 + x[j] : 0.0;
    }
  };
  auto put_zero = [&](int slot) {
#pragma unroll
    for (int j = 0; j < CH; ++j) tile[slot][w][j * 64 + l] = 0.0;
  };
  auto zero = [&](double (&x)[CH]) {
#pragma unroll
    for (int j = 0; j < CH; ++j) x[j] = 0.0;
  };

  double rr0[CH], vr[CH], v2r[CH], rrpost[CH], vrbar[CH], rrbar[CH], rhob[CH];
  R dzr[CH];
  unsigned mix[CH], any = 0;
  stage_sd(0, SD_RR);
  stage_sr(1, SR_VTRR);
  stage_sr(2, SR_VTNR);
  stage_sr(3, SR_RHO);
  stage(4, a.pf);
  for (int e = int(threadIdx.x); e < count; e += 64 * kScrW) {
    const int cc = min(c0 + e % kScrW, a.ncol - 1);
    tile[5][e % kScrW][e / kScrW] = double(value(a.f[F_DZ][TEMPO_IDX_STATE(a, cc, e / kScrW)]));
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int k = j * 64 + l;
    const unsigned pf = k < q.nzc ? unsigned(tile[4][w][k]) : 0u;
    any |= pf;
    mix[j] = pf & PF_SNOWMIX;
    dzr[j] = k < q.nzc ? R(S_t<R>(tile[5][w][k])) : R(1.0);
    q.odz[j] = 1.0 / double(value(dzr[j]));
    q.orho[j] = k < q.nzc ? 1.0 / tile[3][w][k] : 0.0;
  }
  any = wv::uor(any);
  if (l == 0) any_w[w] = any;
  const double dt = a.dt;
  const double pb_rain = live ? g.pbar[c] : 0.0, pb_graupel = live ? g.pbar[a.ncol + c] : 0.0,
               pb_snow = live ? g.pbar[2 * size_t(a.ncol) + c] : 0.0,
               pb_ice = live ? g.pbar[3 * size_t(a.ncol) + c] : 0.0;
  // CFL substeps and ktop from filled speeds (working precision)
  auto cfl = [&](auto vmaxf, int& steps, int& ktop) {
    int st = 1, kt = 1;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int k = j * 64 + l;
      if (k >= q.nzc) continue;
      const R vmax = vmaxf(j);
      if (vmax > R(1.e-3)) {
        kt = max(kt, k + 1);
        const R dz_by_vt = dzr[j] / vmax;
        st = max(st, int(R(dt) / dz_by_vt + R(1.0)));
      }
    }
    steps = wv::imax(st);
    ktop = wv::imax(kt);
    if (ktop == q.nzc) ktop = q.nzc - 1;
  };

  // rain forward values for the snow adjoint
  int rsrc[CH];
  unsigned long long rm[CH];
  int r_steps = 1, r_ktop = 1;
  get(0, rr0);
  zero(rhob);
  zero(vrbar);
  zero(rrbar);
  zero(vr);
  zero(v2r);
#pragma unroll
  for (int j = 0; j < CH; ++j) rrpost[j] = rr0[j];
  if (any & PF_QR) {
    double raw1[CH], raw2[CH];
    get(1, raw1);
    get(2, raw2);
    wave_fill_src(rr0, q.nzc, rsrc, rm);
    wave_gather(raw1, rsrc, vr);
    wave_gather(raw2, rsrc, v2r);
    cfl([&](int j) { return mx(R(vr[j]), R(v2r[j])); }, r_steps, r_ktop);
    const double ost = 1.0 / double(r_steps);
    for (int n = 0; n < r_steps; ++n) {
      double sed[CH];
#pragma unroll
      for (int j = 0; j < CH; ++j) sed[j] = vr[j] * rrpost[j];
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const double up = wv::above(sed, j);
        const int k = j * 64 + l;
        if (k < q.nzc && (k == q.top || k <= r_ktop - 1)) {
          const double flux = (k == q.top) ? -sed[j] : (up - sed[j]);
          const double v = rrpost[j] + flux * q.odz[j] * dt * ost;
          rrpost[j] = v > kR1 ? v : kR1;
        }
      }
    }
  }
  __syncthreads();
  unsigned any_b = 0;  // of the block's columns
#pragma unroll
  for (int i = 0; i < kScrW; ++i) any_b |= any_w[i];

  // ---- cloud ----
  if (any_b & PF_QC) {
    stage_sd(0, SD_RC);
    stage_sd(1, SD_NC);
    stage_sr(2, SR_VTRC);
    stage_sr(3, SR_VTNC);
    stage_ub(4, 8);
    stage_ub(5, 9);
    __syncthreads();
    if (any & PF_QC) {
      double xc[CH];
      get(0, xc);
      int kt = 1;
      R hgt = R(0.0);
      for (int k = 0; k < q.nzc - 1; ++k) {
        if (wv::at_level(xc, k) > kR2) kt = k + 1;
        hgt = hgt + wv::at_level(dzr, k);
        if (hgt > R(500.0)) break;
      }
      for (int f2 = 0; f2 < 2; ++f2) {
        double x0[CH], raw[CH], vt[CH], tb[CH], xb[CH], vb[CH];
        get(f2, x0);
        get(2 + f2, raw);
        get(4 + f2, tb);
#pragma unroll
        for (int j = 0; j < CH; ++j) vt[j] = (j * 64 + l < kt) ? raw[j] : 0.0;
        zero(xb);
        zero(vb);
        wave_sed_adjoint(q, x0, vt, tb, f2 ? kR2 : kR1, 1, 1, kt, 0.0, xb, vb, rhob);
#pragma unroll
        for (int j = 0; j < CH; ++j)
          if (j * 64 + l >= kt) vb[j] = 0.0;
        put(f2, xb);
        put(2 + f2, vb);
      }
    } else {
      for (int i = 0; i < 4; ++i) put_zero(i);
    }
    __syncthreads();
    flush(0, AZ_RC);
    flush(1, AZ_NC);
    flush(2, AZ_VTRC);
    flush(3, AZ_VTNC);
    __syncthreads();
  } else {
    clear_z(AZ_RC);
    clear_z(AZ_NC);
    clear_z(AZ_VTRC);
    clear_z(AZ_VTNC);
  }
  // ---- ice: one application with steps = substeps ----
  if (any_b & PF_QI) {
    stage_sd(0, SD_RI);
    stage_sd(1, SD_NI);
    stage_sr(2, SR_VTRI);
    stage_sr(3, SR_VTNI);
    stage_ub(4, 6);
    stage_ub(5, 7);
    __syncthreads();
    if (any & PF_QI) {
      double xi[CH], raw1[CH], raw2[CH], v1[CH], v2[CH];
      int src[CH];
      unsigned long long m[CH];
      get(0, xi);
      get(2, raw1);
      get(3, raw2);
      wave_fill_src(xi, q.nzc, src, m);
      wave_gather(raw1, src, v1);
      wave_gather(raw2, src, v2);
      int st, kt;
      cfl([&](int j) { return R(v1[j]); }, st, kt);
      for (int f2 = 0; f2 < 2; ++f2) {
        double x0[CH], tb[CH], xb[CH], vb[CH], acc[CH];
        get(f2, x0);
        get(4 + f2, tb);
        zero(xb);
        zero(vb);
        wave_sed_adjoint(q, x0, f2 ? v2 : v1, tb, f2 ? kR2 : kR1, 1, st, kt, f2 ? 0.0 : pb_ice, xb, vb, rhob);
        put(f2, xb);
        zero(acc);
        wave_scatter(vb, src, m, row, q.nzc, acc);
        put(2 + f2, acc);
      }
    } else {
      for (int i = 0; i < 4; ++i) put_zero(i);
    }
    __syncthreads();
    flush(0, AZ_RI);
    flush(1, AZ_NI);
    flush(2, AZ_VTRI);
    flush(3, AZ_VTNI);
    __syncthreads();
  } else {
    clear_z(AZ_RI);
    clear_z(AZ_NI);
    clear_z(AZ_VTRI);
    clear_z(AZ_VTNI);
  }
  // ---- snow: speed mixed with rain where snow melts ----
  if (any_b & PF_QS) {
    stage_sd(0, SD_RS);
    stage_sr(1, SR_VTS);
    stage_ub(2, 5);
    __syncthreads();
    if (any & PF_QS) {
      double xs[CH], raw[CH], vraw[CH], v1[CH], tb[CH];
      int src[CH];
      unsigned long long m[CH];
      get(0, xs);
      get(1, raw);
      get(2, tb);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        R v = R(raw[j]);
        if (mix[j]) {
          const R sr_ = R(xs[j] / (xs[j] + rrpost[j]));
          v = v * sr_ + (R(1.0) - sr_) * R(vr[j]);
        }
        vraw[j] = double(value(v));
      }
      wave_fill_src(xs, q.nzc, src, m);
      wave_gather(vraw, src, v1);
      int st, kt;
      cfl([&](int j) { return R(v1[j]); }, st, kt);
      double xb[CH], vb[CH], acc[CH], zs[CH], zv[CH];
      zero(xb);
      zero(vb);
      wave_sed_adjoint(q, xs, v1, tb, kR1, st, st, kt, pb_snow, xb, vb, rhob);
      zero(acc);
      wave_scatter(vb, src, m, row, q.nzc, acc);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        zs[j] = xb[j];
        zv[j] = 0.0;
        const double vbk = acc[j];
        if (vbk == 0.0) continue;
        if (mix[j]) {
          const double rs = xs[j], rr = rrpost[j], den = rs + rr;
          const double sr_ = rs / den;
          zv[j] = vbk * sr_;
          vrbar[j] += vbk * (1.0 - sr_);
          const double srb = vbk * (raw[j] - vr[j]);
          zs[j] += srb * rr / (den * den);
          rrbar[j] += -srb * rs / (den * den);
        } else {
          zv[j] = vbk;
        }
      }
      put(0, zs);
      put(1, zv);
    } else {
      put_zero(0);
      put_zero(1);
    }
    __syncthreads();
    flush(0, AZ_RS);
    flush(1, AZ_VTS);
    __syncthreads();
  } else {
    clear_z(AZ_RS);
    clear_z(AZ_VTS);
  }
  // ---- graupel ----
  if (any_b & PF_QG) {
    const int fms[3] = {SD_RG, SD_NG, SD_RB}, ten[3] = {2, 3, 4};
    for (int i = 0; i < 3; ++i) stage_sd(i, fms[i]);
    stage_sr(3, SR_VTRG);
    stage_sr(4, SR_VTNG);
    __syncthreads();
    double raw1[CH], raw2[CH], v1[CH], v2[CH], zv[CH];
    int src[CH];
    unsigned long long m[CH];
    int st = 1, kt = 1;
    const bool on = any & PF_QG;
    if (on) {
      double xg[CH];
      get(0, xg);
      get(3, raw1);
      get(4, raw2);
      wave_fill_src(xg, q.nzc, src, m);
      wave_gather(raw1, src, v1);
      wave_gather(raw2, src, v2);
      cfl([&](int j) { return R(v1[j]); }, st, kt);
    } else {
      for (int i = 0; i < 5; ++i) put_zero(i);
    }
    const double rb_lim = kM3ToL * kR1 / 800.0;
    const double lims[3] = {kR1, kR2, rb_lim};
    for (int f3 = 0; f3 < 3; ++f3) {
      stage_ub(5, ten[f3]);
      __syncthreads();
      if (on) {
        double x0[CH], tb[CH], xb[CH], vb[CH], acc[CH];
        get(f3, x0);
        get(5, tb);
        zero(xb);
        zero(vb);
        wave_sed_adjoint(q, x0, f3 == 1 ? v2 : v1, tb, lims[f3], st, st, kt, f3 == 0 ? pb_graupel : 0.0, xb, vb, rhob);
        put(f3, xb);
        zero(acc);
        wave_scatter(vb, src, m, row, q.nzc, acc);
        if (f3 == 1) {
          put(4, acc);
        } else {  // mass and volume share the mass's speed
#pragma unroll
          for (int j = 0; j < CH; ++j) zv[j] = f3 == 0 ? acc[j] : zv[j] + acc[j];
          put(3, zv);
        }
      }
      __syncthreads();
    }
    flush(0, AZ_RG);
    flush(1, AZ_NG);
    flush(2, AZ_RB);
    flush(3, AZ_VTRG);
    flush(4, AZ_VTNG);
    __syncthreads();
  } else {
    clear_z(AZ_RG);
    clear_z(AZ_NG);
    clear_z(AZ_RB);
    clear_z(AZ_VTRG);
    clear_z(AZ_VTNG);
  }
  // ---- rain: final masses and filled speed carry the snow cotangents ----
  if (any_b & PF_QR) {
    stage_sd(0, SD_NR);
    stage_ub(1, 0);
    stage_ub(2, 1);
    __syncthreads();
    if (any & PF_QR) {
      for (int f2 = 0; f2 < 2; ++f2) {
        double x0[CH], tb[CH], xb[CH], vb[CH], acc[CH];
        get(0, x0);
        get(1 + f2, tb);
#pragma unroll
        for (int j = 0; j < CH; ++j) {
          x0[j] = f2 ? x0[j] : rr0[j];
          xb[j] = f2 ? 0.0 : rrbar[j];
          vb[j] = f2 ? 0.0 : vrbar[j];
        }
        wave_sed_adjoint(q, x0, f2 ? v2r : vr, tb, f2 ? kR2 : kR1, r_steps, r_steps, r_ktop, f2 ? 0.0 : pb_rain, xb,
                         vb, rhob);
        put(f2 ? 0 : 3, xb);
        zero(acc);
        wave_scatter(vb, rsrc, rm, row, q.nzc, acc);
        put(f2 ? 5 : 4, acc);
      }
    } else {
      put(3, rrbar);
      put_zero(0);
      put_zero(4);
      put_zero(5);
    }
    put(1, rhob);
    __syncthreads();
    flush(3, AZ_RR);
    flush(0, AZ_NR);
    flush(4, AZ_VTRR);
    flush(5, AZ_VTNR);
    flush(1, AZ_RHO);
  } else {
    put(3, rrbar);
    put(1, rhob);
    __syncthreads();
    flush(3, AZ_RR);
    flush(1, AZ_RHO);
    clear_z(AZ_NR);
    clear_z(AZ_VTRR);
    clear_z(AZ_VTNR);
  }
}

// Copies an adjoint step needs: the working-precision and FP64 scratch planes
// after phase A (used for nz > 128 only), and the post-sedimentation tendency
// values (NULL where nothing overwrites them).
struct AdjSnap {
  void* sr_a;  // sr_bytes
  void* sd_a;  // sd_bytes
  void* sd_b;  // sd_bytes (holds 10 FP64 planes of the post-sedimentation tendencies)
};

// The passes of one adjoint: all tangent passes and S^T.  The state is out of place: a.f holds the
// packed inputs (duals, zero tangents: the passes seed what they read), a.fa
// the state after the initial checks (phase A's output); no pass stores a new
// state.
template <class D>
hipError_t adjoint_passes(const StepArgs<D>& a, AdjArgs g, Dual<double>* vtbuf, size_t sr_bytes,
                          size_t sd_bytes, AdjSnap snap, const AdjLocal<D>& scr, const bool* have_x, hipStream_t s) {
  const unsigned gc = unsigned((a.ncol + 255) / 256);
  const dim3 g2(gc, unsigned(a.nz));
  hipError_t e;
  auto cp = [&](void* dst, const void* src, size_t n) { return hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToDevice, s); };
  auto phase_pre_a = [&]() {
    launch_prepass(a, s);
    hipLaunchKernelGGL(k_phase_a<D>, level_grid(a, 256), dim3(256), 0, s, a);
  };
  // the final update's passes skip the levels without output cotangents
  hipLaunchKernelGGL(k_adj_level_zero<D>, dim3(unsigned((a.nz + 255) / 256)), dim3(256), 0, s, a, g);
  hipLaunchKernelGGL(k_adj_level_flags<D>, g2, dim3(256), 0, s, a, g);

  // tangent-free forward.  Its sedimentation on the values, one wavefront
  // per column (the tangents are zero in this pass), writes only the ten
  // tendency planes, which S^T does not read and whose values the later passes
  // want as they are, so the scratch after A needs no snapshot.  The
  // lane-per-column form (nz > 128) uses state planes as work space: the
  // scratch after A is snapshotted and restored before S^T.
  const bool wave_b = a.nz <= kSedLevels;
  phase_pre_a();
  if (!wave_b) {
    if ((e = cp(snap.sr_a, a.sr, sr_bytes)) != hipSuccess) return e;
    if ((e = cp(snap.sd_a, a.sd, sd_bytes)) != hipSuccess) return e;
  }
  if (wave_b)
    launch_phase_b_wave(a, s);
  else
    hipLaunchKernelGGL(k_phase_b<D>, dim3(unsigned((a.ncol + 127) / 128)), dim3(128), 0, s, a, vtbuf);
  // the post-sedimentation tendency values stay in the scratch for the local
  // passes, or are copied where these or the restored snapshot overwrite it
  double* post = static_cast<double*>(snap.sd_b);
  g.post = post;
  if (post) hipLaunchKernelGGL(k_adj_keep_post<D>, g2, dim3(256), 0, s, a, post);
  // passes seeded on the post-sedimentation tendencies.  Without prognostic
  // graupel number and volume the final update does not read their
  // tendencies, so those cotangents are zero and need no pass.
  const bool ngqb = a.f[F_NG] && a.f[F_QB];
  AdjDirs ms{};
  for (int m = 0; m < 10; ++m) {
    if (!ngqb && (SD_QRTEN + m == SD_NGTEN || SD_QRTEN + m == SD_QBTEN)) {
      double* ub = g.ubar + size_t(m) * a.plane;
      hipLaunchKernelGGL(k_adj_zero<double>, dim3(unsigned((a.plane + 255) / 256)), dim3(256), 0, s, ub, a.plane);
      continue;
    }
    ms.id[ms.n++] = m;
  }
  hipLaunchKernelGGL(k_adj_upass<D>, dim3(gc, unsigned(a.nz), unsigned(ms.n)), dim3(256), 0, s, a, g, ms);
  // S^T on the values after phase A
  if (!wave_b) {
    if ((e = cp(a.sr, snap.sr_a, sr_bytes)) != hipSuccess) return e;
    if ((e = cp(a.sd, snap.sd_a, sd_bytes)) != hipSuccess) return e;
  }
  const dim3 gw(unsigned((a.ncol + kScrW - 1) / kScrW));
  if (a.nz <= 64)
    hipLaunchKernelGGL((k_adj_sed_wave<D, 1>), gw, dim3(64 * kScrW), 0, s, a, g);
  else if (wave_b)
    hipLaunchKernelGGL((k_adj_sed_wave<D, 2>), gw, dim3(64 * kScrW), 0, s, a, g);
  else
    hipLaunchKernelGGL(k_adj_sedimentation<D>, dim3(unsigned((a.ncol + 63) / 64)), dim3(64), 0, s, a, g);
  // the local passes, as many directions in a launch and then as many points
  // as the scratch holds.  The count of listed points stays on the device:
  // launches past it end at once.  The pre-pass results (column flags,
  // heights) depend on values only and stay from the forward.
  AdjDirs xs{};
  for (int i = 0; i < AX_N; ++i)
    if (have_x[i]) xs.id[xs.n++] = i;
  if (xs.n == 0) return hipGetLastError();
  hipLaunchKernelGGL(k_adj_point_list<D>, g2, dim3(256), 0, s, a, g, xs);
  const size_t n3 = size_t(a.ncol) * a.nz;
  const size_t together = std::min(size_t(xs.n), scr.room);
  size_t points = std::min(scr.room / together, n3);
  if (points >= 64 && points < n3) points = points / 64 * 64;
  for (int j = 0; j < xs.n; j += int(together)) {
    AdjDirs d{};
    for (int i = j; i < xs.n && i < j + int(together); ++i) d.id[d.n++] = xs.id[i];
    const dim3 gl(unsigned((points + 255) / 256), 1, unsigned(d.n));
    for (size_t first = 0; first < n3; first += points) {
      hipLaunchKernelGGL(k_adj_local_a<D>, gl, dim3(256), 0, s, a, g, scr, d, unsigned(first), unsigned(points));
      hipLaunchKernelGGL(k_adj_local_c<D>, gl, dim3(256), 0, s, a, g, scr, d, unsigned(first), unsigned(points));
    }
  }
  return hipGetLastError();
}

}  // namespace tempo
