// C ABI of the TEMPO column step (declared in include/tempo_hip.h).
#include "tempo_hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "tempo_capi_internal.hpp"
#include "tempo_host.hpp"
#include "tempo_step.hpp"
#include "tempo_adjoint.hpp"
#include "tempo_adjoint_wave.hpp"

namespace tempo {
// defined in tempo_step_f32.hip / tempo_step_f64.hip / tempo_tables.hip
hipError_t launch_step(const StepArgs<float>& a, const LaunchCfg& lc, double* vtbuf, hipStream_t s, hipEvent_t* ev);
hipError_t launch_step(const StepArgs<double>& a, const LaunchCfg& lc, double* vtbuf, hipStream_t s, hipEvent_t* ev);
hipError_t launch_step_sig(const StepArgs<float>& a, const LaunchCfg& lc, double* vtbuf, hipStream_t s);
hipError_t launch_step_sig(const StepArgs<double>& a, const LaunchCfg& lc, double* vtbuf, hipStream_t s);
hipError_t launch_step_tlm(const StepArgs<Dual<float>>& a, const LaunchCfg& lc, Dual<double>* vtbuf, hipStream_t s);
hipError_t launch_step_tlm(const StepArgs<Dual<double>>& a, const LaunchCfg& lc, Dual<double>* vtbuf, hipStream_t s);
template <class R>
hipError_t launch_check_update(const CheckArgs<R>& g, int which, hipStream_t s);
template <class R>
hipError_t launch_surface_emissions(R* nwfa, const R* nwfa2d, int ni, int nj, long long ldk, long long ldj,
                                    long long d2ldj, int k, double dt, hipStream_t s);
hipError_t launch_adjoint(const StepArgs<Dual<float>>& a, const AdjArgs& g, Dual<double>* vtbuf, size_t sr_bytes,
                          size_t sd_bytes, AdjSnap snap, const AdjLocal<Dual<float>>& scr, const bool* have_x,
                          hipStream_t s);
hipError_t launch_adjoint(const StepArgs<Dual<double>>& a, const AdjArgs& g, Dual<double>* vtbuf, size_t sr_bytes,
                          size_t sd_bytes, AdjSnap snap, const AdjLocal<Dual<double>>& scr, const bool* have_x,
                          hipStream_t s);
template <class T>
hipError_t launch_to_compact_n(const PlaneBatch<T, double>& b, int n, const DualGeom& g, hipStream_t s);
template <class T>
hipError_t launch_from_compact_n(const PlaneBatch<double, T>& b, int n, const DualGeom& g, hipStream_t s);
template <class T>
hipError_t launch_dual_pack_n(const DualBatch<T>& b, int n, const DualGeom& g, hipStream_t s);
template <class T>
hipError_t launch_dual_unpack_n(const DualBatch<T>& b, int n, const DualGeom& g, const int* nlev, hipStream_t s);
hipError_t launch_table_qg(const double*, const double*, const double*, const double*, double*, hipStream_t);
hipError_t launch_table_qs(const double*, const double*, const double*, const double*, double*, hipStream_t);
hipError_t launch_table_fz(const double*, const double*, const double*, const double*, double, const double*,
                           const double*, const double*, const double*, const double*, double*, hipStream_t);
template <class T>
hipError_t launch_pack(const double* src, size_t n, int narr, T* dst, hipStream_t s);
}  // namespace tempo

using namespace tempo;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                                     \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess) return fail(TEMPO_HIP_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

// Owns one device allocation.  Move-only: a copy would free the same pointer
// twice (containers of DevBuf move their elements when they grow).
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept : p(o.p), bytes(o.bytes) {
    o.p = nullptr;
    o.bytes = 0;
  }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) {
      if (p) (void)hipFree(p);
      p = o.p;
      bytes = o.bytes;
      o.p = nullptr;
      o.bytes = 0;
    }
    return *this;
  }
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  hipError_t ensure(size_t n) {
    if (n <= bytes) return hipSuccess;
    if (p) {
      hipError_t e = hipFree(p);
      if (e != hipSuccess) return e;
      p = nullptr;
      bytes = 0;
    }
    hipError_t e = hipMalloc(&p, n);
    if (e == hipSuccess) bytes = n;
    return e;
  }
  template <class T>
  T* as() const { return static_cast<T*>(p); }
};
static_assert(!std::is_copy_constructible<DevBuf>::value && std::is_nothrow_move_constructible<DevBuf>::value,
              "DevBuf owns its allocation");

template <class T>
hipError_t upload(DevBuf& b, const std::vector<T>& v) {
  hipError_t e = b.ensure(v.size() * sizeof(T));
  if (e != hipSuccess) return e;
  return hipMemcpy(b.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
}

// Const<double> -> Const<float>: the R-typed members form one contiguous
// prefix followed by the int members.
void narrow(const Const<double>& d, Const<float>& f) {
  static_assert(sizeof(LaneConst<double>) == 2 * sizeof(LaneConst<float>), "LaneConst layout");
  const double* src = reinterpret_cast<const double*>(&d);
  float* dst = reinterpret_cast<float*>(&f);
  const size_t nr = size_t(reinterpret_cast<const double*>(&d.nic2) - src);
  for (size_t i = 0; i < nr; ++i) dst[i] = float(src[i]);
  std::memcpy(&f.nic2, &d.nic2, sizeof(int) * 10);
}

bool read_file(const std::string& path, std::vector<char>& out, std::string& err) {
  FILE* fp = std::fopen(path.c_str(), "rb");
  if (!fp) {
    err = "cannot open " + path;
    return false;
  }
  std::fseek(fp, 0, SEEK_END);
  long n = std::ftell(fp);
  std::fseek(fp, 0, SEEK_SET);
  out.resize(size_t(n));
  size_t got = n > 0 ? std::fread(out.data(), 1, size_t(n), fp) : 0;
  std::fclose(fp);
  if (got != size_t(n)) {
    err = "short read " + path;
    return false;
  }
  return true;
}

template <class T>
T bswap(T v) {
  T r;
  const unsigned char* s = reinterpret_cast<const unsigned char*>(&v);
  unsigned char* d = reinterpret_cast<unsigned char*>(&r);
  for (size_t i = 0; i < sizeof(T); ++i) d[i] = s[sizeof(T) - 1 - i];
  return r;
}

// one host copy of the host-array staging
struct Piece {
  char* dst;
  const char* src;
  size_t n;
};

// Host threads for the host-array staging: run() splits the bytes of a list
// of copies evenly over the pool's threads and the calling thread and
// returns when every copy is done.
class CopyPool {
 public:
  explicit CopyPool(unsigned threads) : nt_(std::max(1u, threads)) {
    for (unsigned i = 1; i < nt_; ++i) th_.emplace_back([this, i] { work(i); });
  }
  ~CopyPool() {
    {
      std::lock_guard<std::mutex> g(m_);
      stop_ = true;
    }
    go_.notify_all();
    for (auto& t : th_) t.join();
  }
  CopyPool(const CopyPool&) = delete;
  CopyPool& operator=(const CopyPool&) = delete;
  unsigned threads() const { return nt_; }
  void run(const std::vector<Piece>& p) {
    size_t total = 0;
    for (const Piece& q : p) total += q.n;
    if (nt_ == 1 || total < (size_t(1) << 20)) {
      share(p, total, 0, 1);
      return;
    }
    {
      std::lock_guard<std::mutex> g(m_);
      job_ = &p;
      total_ = total;
      pending_ = nt_ - 1;
      ++gen_;
    }
    go_.notify_all();
    share(p, total, 0, nt_);
    std::unique_lock<std::mutex> l(m_);
    done_.wait(l, [this] { return pending_ == 0; });
  }

 private:
  // thread id of n copies bytes [total*id/n, total*(id+1)/n) of the list
  static void share(const std::vector<Piece>& p, size_t total, unsigned id, unsigned n) {
    const size_t a = total * id / n, b = total * (id + 1) / n;
    size_t at = 0;
    for (const Piece& q : p) {
      if (at >= b) break;
      const size_t lo = std::max(a, at), hi = std::min(b, at + q.n);
      if (lo < hi) std::memcpy(q.dst + (lo - at), q.src + (lo - at), hi - lo);
      at += q.n;
    }
  }
  void work(unsigned id) {
    unsigned seen = 0;
    for (;;) {
      const std::vector<Piece>* job;
      size_t total;
      {
        std::unique_lock<std::mutex> l(m_);
        go_.wait(l, [&] { return stop_ || gen_ != seen; });
        if (stop_) return;
        seen = gen_;
        job = job_;
        total = total_;
      }
      share(*job, total, id, nt_);
      std::lock_guard<std::mutex> g(m_);
      if (--pending_ == 0) done_.notify_one();
    }
  }
  unsigned nt_;
  std::vector<std::thread> th_;
  std::mutex m_;
  std::condition_variable go_, done_;
  const std::vector<Piece>* job_ = nullptr;
  size_t total_ = 0;
  unsigned pending_ = 0, gen_ = 0;
  bool stop_ = false;
};

}  // namespace

struct tempo_hip_ctx {
  tempo_hip_cfg cfg;
  int device = 0;
  Const<double> cd;
  Const<float> cf;
  DevBuf cd_dev, cf_dev;  // the constants in device memory, one copy per context
  // reference-order FP64 tables
  DevBuf qg_ref, qs_ref, fz_ref;
  // gather layouts
  DevBuf qg64, qs64, fzr64, fzc64, qg32, qs32, fzr32, fzc32;
  DevBuf ccn;  // float slice (7,9,7)
  DevBuf efrw64, efsw64, wev64, iaus64, efrw32, efsw32, wev32, iaus32;
  // scratch
  DevBuf sr, sd, pf, cf_, precip, ksub, vtbuf, kmelt, radar;
  DevBuf semiw;  // semi-Lagrangian sedimentation work (allocated only with semi_sedi_flag)
  DevBuf tl_state, tl_diag;  // dual (value, tangent) copies for the tangent-linear step
  DevBuf adj_in, adj_local, adj_mem;  // adjoint: packed inputs, local passes' scratch, cotangent/Jacobian planes
  DevBuf adj_snap;                  // adjoint: post-sedimentation tendencies (and scratch after A)
  int last_ncol = 0;
  void* last_ksub = nullptr;  // substep counts of the last run (its scratch)
  void* last_vt = nullptr;    // its wide sedimentation planes
  // host-array staging: device copies of the caller's arrays (FP64, and
  // their FP32 working copies); pinned slab buffers, two for uploads and
  // three for downloads, with their events; the compute, upload and
  // download streams of host runs; the copy threads
  std::vector<DevBuf> stage, stage32;
  DevBuf stage_land, stage_nlev;
  void* pin_up[2] = {nullptr, nullptr};
  void* pin_dn[3] = {nullptr, nullptr, nullptr};
  size_t pin_up_bytes = 0, pin_dn_bytes = 0;
  hipEvent_t ev_up[2] = {nullptr, nullptr};
  hipEvent_t ev_dn[3] = {nullptr, nullptr, nullptr};
  hipEvent_t ev_step = nullptr;
  hipStream_t host_stream = nullptr, up_stream = nullptr, down_stream = nullptr;
  std::unique_ptr<CopyPool> pool;
  double build_ms = 0.0;
  LaunchCfg launch[2];  // [FP32, FP64]
  // per-phase timing: 5 events per profiled run
  bool profile = false;
  std::vector<hipEvent_t> events;
  ~tempo_hip_ctx() {
    for (auto e : events) (void)hipEventDestroy(e);
    for (hipStream_t st : {host_stream, up_stream, down_stream})
      if (st) (void)hipStreamSynchronize(st);
    for (void* b : pin_up)
      if (b) (void)hipHostFree(b);
    for (void* b : pin_dn)
      if (b) (void)hipHostFree(b);
    for (hipEvent_t e : ev_up)
      if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : ev_dn)
      if (e) (void)hipEventDestroy(e);
    if (ev_step) (void)hipEventDestroy(ev_step);
    for (hipStream_t st : {host_stream, up_stream, down_stream})
      if (st) (void)hipStreamDestroy(st);
  }
};

extern "C" {

void tempo_hip_cfg_default(tempo_hip_cfg* c) {
  std::memset(c, 0, sizeof(*c));
  c->aerosolaware_flag = 1;
  c->hailaware_flag = 1;
  c->cloud_condensation_flag = 1;
  c->nc_option = 0;
  c->nc_value = 100.e6;
  c->refl10cm_flag = 1;
  c->re_cloud_flag = 1;
  c->re_ice_flag = 1;
  c->re_snow_flag = 1;
  c->max_hail_diameter_flag = 1;
}

const char* tempo_hip_last_error(void) { return g_err.c_str(); }

int tempo_hip_set_run_cfg(tempo_hip_ctx* x, const tempo_hip_cfg* cfg) {
  if (!x || !cfg) return fail(TEMPO_HIP_E_ARG, "tempo_hip_set_run_cfg: NULL argument");
  if (cfg->aerosolaware_flag != x->cfg.aerosolaware_flag || cfg->hailaware_flag != x->cfg.hailaware_flag)
    return fail(TEMPO_HIP_E_ARG, "aerosolaware_flag and hailaware_flag are fixed at tempo_hip_init");
  x->cfg = *cfg;
  return TEMPO_HIP_OK;
}

void tempo_hip_finalize(tempo_hip_ctx* ctx) { delete ctx; }

double tempo_hip_table_build_ms(tempo_hip_ctx* ctx) { return ctx ? ctx->build_ms : 0.0; }

}  // extern "C"

namespace {

int upload_small_tables(tempo_hip_ctx* x) {
  HostBins hb;
  Const<double> c;
  build_const(c, hb, x->cfg.hailaware_flag != 0);
  SmallTables t;
  build_small_tables(c, hb, t);
  auto both = [&](const std::vector<double>& v, DevBuf& d64, DevBuf& d32) -> hipError_t {
    hipError_t e = upload(d64, v);
    if (e != hipSuccess) return e;
    std::vector<float> f(v.begin(), v.end());
    return upload(d32, f);
  };
  HIP_TRY(both(t.efrw, x->efrw64, x->efrw32));
  HIP_TRY(both(t.efsw, x->efsw64, x->efsw32));
  HIP_TRY(both(t.tnc_wev, x->wev64, x->wev32));
  std::vector<double> iaus(t.tps_iaus);
  iaus.insert(iaus.end(), t.tni_iaus.begin(), t.tni_iaus.end());
  iaus.insert(iaus.end(), t.tpi_ide.begin(), t.tpi_ide.end());
  HIP_TRY(both(iaus, x->iaus64, x->iaus32));
  return TEMPO_HIP_OK;
}

int build_tables_gpu(tempo_hip_ctx* x) {
  TableFactors f;
  build_table_factors(f);
  DevBuf nr, qga, qgng, qsa, qsns, massr, massc, probr, probc, nc, tnc, rr, rc;
  HIP_TRY(upload(nr, f.n_r));
  HIP_TRY(upload(qga, f.qg_a));
  HIP_TRY(upload(qgng, f.qg_ng));
  HIP_TRY(upload(qsa, f.qs_a));
  HIP_TRY(upload(qsns, f.qs_ns));
  HIP_TRY(upload(massr, f.fz_massr));
  HIP_TRY(upload(massc, f.fz_massc));
  HIP_TRY(upload(probr, f.fz_prob_r));
  HIP_TRY(upload(probc, f.fz_prob_c));
  HIP_TRY(upload(nc, f.fz_nc));
  HIP_TRY(upload(tnc, f.fz_t_nc));
  HIP_TRY(upload(rr, f.r_r));
  HIP_TRY(upload(rc, f.r_c));
  HIP_TRY(x->qg_ref.ensure(kNQgArr * kNQg1 * sizeof(double)));
  HIP_TRY(x->qs_ref.ensure(kNQsArr * kNQs1 * sizeof(double)));
  HIP_TRY(x->fz_ref.ensure((kNFzRArr * kNFzR1 + kNFzCArr * kNFzC1) * sizeof(double)));
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  HIP_TRY(hipEventRecord(e0, nullptr));
  HIP_TRY(launch_table_qg(qga.as<double>(), qgng.as<double>(), nr.as<double>(), rr.as<double>(),
                          x->qg_ref.as<double>(), nullptr));
  HIP_TRY(launch_table_qs(qsa.as<double>(), qsns.as<double>(), nr.as<double>(), rr.as<double>(),
                          x->qs_ref.as<double>(), nullptr));
  HIP_TRY(launch_table_fz(nr.as<double>(), probr.as<double>(), massr.as<double>(), rr.as<double>(), f.fz_xm0g,
                          nc.as<double>(), probc.as<double>(), massc.as<double>(), tnc.as<double>(), rc.as<double>(),
                          x->fz_ref.as<double>(), nullptr));
  HIP_TRY(hipEventRecord(e1, nullptr));
  HIP_TRY(hipEventSynchronize(e1));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
  x->build_ms = ms;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return TEMPO_HIP_OK;
}

int read_tables(tempo_hip_ctx* x, const std::string& dir) {
  struct Item {
    const char* name;
    DevBuf* dst;
    size_t n;
  } items[3] = {{"freeze_water_data_tempo_v3", &x->fz_ref, kNFzRArr * kNFzR1 + kNFzCArr * kNFzC1},
                {"qr_acr_qs_data_tempo_v3", &x->qs_ref, kNQsArr * kNQs1},
                {"qr_acr_qg_data_tempo_v3", &x->qg_ref, kNQgArr * kNQg1}};
  for (auto& it : items) {
    std::vector<char> raw;
    std::string err;
    if (!read_file(dir + "/" + it.name, raw, err)) return fail(TEMPO_HIP_E_TABLE, err);
    if (raw.size() != it.n * sizeof(double))
      return fail(TEMPO_HIP_E_TABLE, std::string(it.name) + ": size " + std::to_string(raw.size()) +
                                         " bytes, expected " + std::to_string(it.n * sizeof(double)));
    std::vector<double> v(it.n);
    const double* src = reinterpret_cast<const double*>(raw.data());
    for (size_t i = 0; i < it.n; ++i) v[i] = bswap(src[i]);
    HIP_TRY(upload(*it.dst, v));
  }
  return TEMPO_HIP_OK;
}

int read_ccn(tempo_hip_ctx* x, const std::string& path) {
  std::vector<char> raw;
  std::string err;
  if (!read_file(path, raw, err)) return fail(TEMPO_HIP_E_TABLE, err);
  if (raw.size() != kNCcn * 4 + 8) return fail(TEMPO_HIP_E_TABLE, path + ": wrong size");
  uint32_t head;
  std::memcpy(&head, raw.data(), 4);
  if (bswap(head) != kNCcn * 4) return fail(TEMPO_HIP_E_TABLE, path + ": bad record marker");
  const float* v = reinterpret_cast<const float*>(raw.data() + 4);
  // slice tnccn_act(:,:,:,3,2) as [k][j][i] (src/module_mp_tempo_main.F90:2246-2266)
  std::vector<float> s(7 * 9 * 7);
  for (int k = 0; k < 7; ++k)
    for (int j = 0; j < 9; ++j)
      for (int i = 0; i < 7; ++i) {
        size_t fo = size_t(i) + 7 * (j + 9 * (k + 7 * (2 + 5 * 1)));
        s[i + 7 * (j + 9 * k)] = bswap(v[fo]);
      }
  HIP_TRY(upload(x->ccn, s));
  return TEMPO_HIP_OK;
}

int pack_tables(tempo_hip_ctx* x) {
  HIP_TRY(x->qg64.ensure(kNQgArr * kNQg1 * sizeof(double)));
  HIP_TRY(x->qs64.ensure(kNQsArr * kNQs1 * sizeof(double)));
  HIP_TRY(x->fzr64.ensure(kNFzRArr * kNFzR1 * sizeof(double)));
  HIP_TRY(x->fzc64.ensure(kNFzCArr * kNFzC1 * sizeof(double)));
  HIP_TRY(x->qg32.ensure(kNQgArr * kNQg1 * sizeof(float)));
  HIP_TRY(x->qs32.ensure(kNQsArr * kNQs1 * sizeof(float)));
  HIP_TRY(x->fzr32.ensure(kNFzRArr * kNFzR1 * sizeof(float)));
  HIP_TRY(x->fzc32.ensure(kNFzCArr * kNFzC1 * sizeof(float)));
  const double* fz = x->fz_ref.as<double>();
  HIP_TRY(launch_pack<double>(x->qg_ref.as<double>(), kNQg1, kNQgArr, x->qg64.as<double>(), nullptr));
  HIP_TRY(launch_pack<double>(x->qs_ref.as<double>(), kNQs1, kNQsArr, x->qs64.as<double>(), nullptr));
  HIP_TRY(launch_pack<double>(fz, kNFzR1, kNFzRArr, x->fzr64.as<double>(), nullptr));
  HIP_TRY(launch_pack<double>(fz + kNFzRArr * kNFzR1, kNFzC1, kNFzCArr, x->fzc64.as<double>(), nullptr));
  HIP_TRY(launch_pack<float>(x->qg_ref.as<double>(), kNQg1, kNQgArr, x->qg32.as<float>(), nullptr));
  HIP_TRY(launch_pack<float>(x->qs_ref.as<double>(), kNQs1, kNQsArr, x->qs32.as<float>(), nullptr));
  HIP_TRY(launch_pack<float>(fz, kNFzR1, kNFzRArr, x->fzr32.as<float>(), nullptr));
  HIP_TRY(launch_pack<float>(fz + kNFzRArr * kNFzR1, kNFzC1, kNFzCArr, x->fzc32.as<float>(), nullptr));
  HIP_TRY(hipDeviceSynchronize());
  return TEMPO_HIP_OK;
}

size_t scratch_plane(size_t ncol, size_t nz) { return (ncol + kScrW - 1) / kScrW * kScrW * size_t(scratch_levels(int(nz))); }

// Byte sizes of the per-point scratch of one step of ncol columns of nz
// levels; br / bw / bd: bytes of one working-precision / wide /
// sedimented-state value (8, 8, 4 or 8 for the plain step, 16 for duals);
// vt_planes: wide planes of the one-lane-per-column sedimentation (3
// fall-speed planes, plus a wide copy of the SD_N planes when these are
// stored narrower); semi: semi-Lagrangian work arrays.
struct ScratchSizes {
  size_t sr, sd, pf, vt, cf, kmelt, precip, ksub, semiw;
  ScratchSizes(size_t ncol, size_t nz, size_t br, size_t bw, size_t bd, size_t vt_planes, bool semi) {
    const size_t plane = scratch_plane(ncol, nz);
    sr = SR_N * plane * br;
    sd = SD_N * plane * bd;
    pf = plane * sizeof(unsigned);
    vt = vt_planes * plane * bw;
    cf = ncol * sizeof(unsigned);
    kmelt = ncol * sizeof(int);
    precip = 5 * ncol * bw;
    ksub = kSubRows * ncol * sizeof(int);
    semiw = semi ? kSemiArrays * (nz + 2) * ncol * bw : 0;
  }
  // the buffers carved in this order from one block, each 256-byte aligned
  static size_t up(size_t b) { return (b + 255) / 256 * 256; }
  size_t total() const {
    return up(sr) + up(sd) + up(pf) + up(vt) + up(cf) + up(kmelt) + up(precip) + up(ksub) + up(semiw);
  }
};

// where one step's scratch lives
struct ScratchPtrs {
  void *sr, *sd, *pf, *vt, *cf, *kmelt, *precip, *ksub, *semiw;
};

// the context's own scratch, grown to the sizes (the defaults cover every step)
int ensure_scratch(tempo_hip_ctx* x, size_t ncol, size_t nz, size_t br = 8, size_t bw = 8, size_t bd = 8,
                   size_t vt_planes = 3 + SD_N) {
  const ScratchSizes z(ncol, nz, br, bw, bd, vt_planes, x->cfg.semi_sedi_flag != 0);
  HIP_TRY(x->sr.ensure(z.sr));
  HIP_TRY(x->sd.ensure(z.sd));
  HIP_TRY(x->pf.ensure(z.pf));
  HIP_TRY(x->vtbuf.ensure(z.vt));
  HIP_TRY(x->cf_.ensure(z.cf));
  HIP_TRY(x->kmelt.ensure(z.kmelt));
  HIP_TRY(x->precip.ensure(z.precip));
  HIP_TRY(x->ksub.ensure(z.ksub));
  if (z.semiw) HIP_TRY(x->semiw.ensure(z.semiw));
  return TEMPO_HIP_OK;
}

// the scratch sizes of one step of a in the context's configuration, on
// more than wave_levels levels with the wide copy of the lane-per-column
// sedimentation
template <class R>
ScratchSizes step_scratch(const tempo_hip_ctx* x, const StepArgs<R>& a, int wave_levels = kSedMaxLevels) {
  using S = S_t<R>;
  using W = W_t<R>;
  using D = Sd_t<R>;
  // the wide copy is needed where the one-lane-per-column sedimentation runs
  // on narrow planes
  const LaunchCfg& lc = x->launch[sizeof(S) == 8 ? 1 : 0];
  const bool lane_sed = !lc.sed_wave || a.nz > wave_levels || x->cfg.semi_sedi_flag;
  const size_t vt_planes = 3 + (sizeof(D) < sizeof(W) && lane_sed ? SD_N : 0);
  return ScratchSizes(size_t(a.ncol), size_t(a.nz), sizeof(R), sizeof(W), sizeof(D), vt_planes,
                      x->cfg.semi_sedi_flag != 0);
}

// Point grouping of a step that sets none.  The FP64 level physics is bound
// by its instructions, so wavefronts full of points with work to do pay for
// finding them at every size (25,000 x 90: 1.85 ms without, 1.56 with; one
// column x 60: 178, 135 us); its final update, bound by memory, only while
// a batch leaves the chip idle (128 columns: 139 us, 130 with; 512: the
// same).  In FP32 both lose by it (100,000 x 90: 2.04 ms, 2.20 with), but
// where the columns fill half a wavefront at most (one column: 78 us, 60; 32:
// 67, 64; 64: 65, 65): four levels then share one.  Duals lose or gain under
// 3 %.
int point_order(bool r64, int ncol) {
  if (r64) return ncol <= 256 ? 3 : 1;
  return ncol <= 32 ? 3 : 0;
}

// scratch, tables, constants and flags of one launch (a.ncol, a.nz set);
// sc: the scratch to use (NULL: the context's own, grown as needed)
template <class R>
int bind_common(tempo_hip_ctx* x, StepArgs<R>& a, double dt, int itimestep, const ScratchPtrs* sc = nullptr) {
  using S = S_t<R>;
  using W = W_t<R>;
  using D = Sd_t<R>;
  ScratchPtrs own;
  if (!sc) {
    const ScratchSizes z = step_scratch(x, a);
    HIP_TRY(x->sr.ensure(z.sr));
    HIP_TRY(x->sd.ensure(z.sd));
    HIP_TRY(x->pf.ensure(z.pf));
    HIP_TRY(x->vtbuf.ensure(z.vt));
    HIP_TRY(x->cf_.ensure(z.cf));
    HIP_TRY(x->kmelt.ensure(z.kmelt));
    HIP_TRY(x->precip.ensure(z.precip));
    HIP_TRY(x->ksub.ensure(z.ksub));
    if (z.semiw) HIP_TRY(x->semiw.ensure(z.semiw));
    own = ScratchPtrs{x->sr.p, x->sd.p, x->pf.p, x->vtbuf.p, x->cf_.p, x->kmelt.p, x->precip.p, x->ksub.p,
                      z.semiw ? x->semiw.p : nullptr};
    sc = &own;
  }
  a.sr = static_cast<R*>(sc->sr);
  a.plane = scratch_plane(size_t(a.ncol), size_t(a.nz));
  a.nzs = scratch_levels(a.nz);
  a.sd = static_cast<D*>(sc->sd);
  a.pf = static_cast<unsigned*>(sc->pf);
  a.cf = static_cast<unsigned*>(sc->cf);
  a.precip = static_cast<W*>(sc->precip);
  a.ksub = static_cast<int*>(sc->ksub);
  x->last_ncol = a.ncol;
  x->last_ksub = sc->ksub;
  x->last_vt = sc->vt;
  const bool r64 = sizeof(S) == 8;
  const int order = x->launch[r64 ? 1 : 0].order;
  a.compact = order >= 0 ? order : IsDual<R>::value ? 0 : point_order(r64, a.ncol);
  a.ccn_lds = x->launch[r64 ? 1 : 0].ccn_lds;
  a.tab.qg = static_cast<const S*>(r64 ? x->qg64.p : x->qg32.p);
  a.tab.qs = static_cast<const S*>(r64 ? x->qs64.p : x->qs32.p);
  a.tab.fzr = static_cast<const S*>(r64 ? x->fzr64.p : x->fzr32.p);
  a.tab.fzc = static_cast<const S*>(r64 ? x->fzc64.p : x->fzc32.p);
  a.tab.ccn = x->ccn.as<float>();
  a.cst = static_cast<const Const<S>*>(r64 ? x->cd_dev.p : x->cf_dev.p);
  for (int i = 0; i < F_NFIELDS; ++i) a.fa[i] = a.fo[i] = a.f[i];  // in place
  a.tab.efrw = static_cast<const S*>(r64 ? x->efrw64.p : x->efrw32.p);
  a.tab.efsw = static_cast<const S*>(r64 ? x->efsw64.p : x->efsw32.p);
  a.tab.tnc_wev = static_cast<const S*>(r64 ? x->wev64.p : x->wev32.p);
  const S* iaus = static_cast<const S*>(r64 ? x->iaus64.p : x->iaus32.p);
  a.tab.tps_iaus = iaus;
  a.tab.tni_iaus = iaus + kNtbI * kNtbI1;
  a.tab.tpi_ide = iaus + 2 * kNtbI * kNtbI1;
  const tempo_hip_cfg& c = x->cfg;
  a.fl.aerosolaware = c.aerosolaware_flag;
  a.fl.hailaware = c.hailaware_flag;
  a.fl.turn_off_micro = c.turn_off_micro_flag;
  a.fl.semi_sedi = c.semi_sedi_flag;
  a.fl.refl_from_melting = c.refl10cm_from_melting_flag;
  a.radar = x->radar.as<Radar>();
  a.kmelt = static_cast<int*>(sc->kmelt);
  a.semiw = c.semi_sedi_flag ? static_cast<W*>(sc->semiw) : nullptr;
  a.fl.cloud_condensation = c.cloud_condensation_flag;
  a.fl.refl10cm = c.refl10cm_flag;
  a.fl.re_cloud = c.re_cloud_flag;
  a.fl.re_ice = c.re_ice_flag;
  a.fl.re_snow = c.re_snow_flag;
  a.fl.max_hail = c.max_hail_diameter_flag;
  a.fl.mvd_r = c.rain_med_vol_diam_flag;
  a.fl.mvd_g = c.graupel_med_vol_diam_flag;
  a.fl.nc_mixing_ratio = c.cloud_number_mixing_ratio_flag;
  a.fl.ml_for_nc = c.ml_for_nc_flag;
  a.fl.ml_for_bl_nc = c.ml_for_bl_nc_flag;
  a.fl.nc_const = c.nc_option == 1 ? kNtCO : (c.nc_option == 2 ? c.nc_value : kNtCL);
  a.dt = dt;
  a.odt = sizeof(S) == 4 ? double(1.0f / float(dt)) : 1.0 / dt;
  a.first_step = itimestep == 1;
  return TEMPO_HIP_OK;
}

void field_ptrs(const tempo_hip_fields* f, void* (&fp)[F_NFIELDS]) {
  void* const v[F_NFIELDS] = {f->t,  f->p,  f->w,  f->dz, f->qv, f->qc,   f->qr,   f->qi, f->qs, f->qg,
                              f->ni, f->nr, f->nc, f->nwfa, f->nifa, f->ng, f->qb, f->th, f->pii};
  for (int i = 0; i < F_NFIELDS; ++i) fp[i] = v[i];
}

void diag_ptrs(const tempo_hip_diags* d, void* (&d2)[D2_N], void* (&d3)[D3_N]) {
  void* const v2[D2_N] = {d->rain_precip, d->ice_liquid_equiv_precip, d->snow_liquid_equiv_precip,
                          d->graupel_liquid_equiv_precip, d->frozen_fraction, d->frz_rain_precip,
                          d->max_hail_diameter_sfc, d->max_hail_diameter_column};
  void* const v3[D3_N] = {d->refl10cm, d->re_cloud, d->re_ice, d->re_snow, d->rain_med_vol_diam,
                          d->graupel_med_vol_diam, d->cloud_number_mixing_ratio};
  for (int i = 0; i < D2_N; ++i) d2[i] = v2[i];
  for (int i = 0; i < D3_N; ++i) d3[i] = v3[i];
}

// sig (device, may be NULL): record the level-local kernels' branch
// signatures there (a signature run; no per-phase timing).  sc: scratch to
// use instead of the context's own (no allocation, no per-phase timing).
template <class R>
int run_impl(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_diags* d, const tempo_hip_dims* dm,
             double dt, int itimestep, hipStream_t s, unsigned* sig = nullptr, const ScratchPtrs* sc = nullptr) {
  StepArgs<R> a;
  std::memset(&a, 0, sizeof(a));
  void* fp[F_NFIELDS];
  field_ptrs(f, fp);
  for (int i = 0; i < F_NFIELDS; ++i) a.f[i] = static_cast<R*>(fp[i]);
  if (d) {
    void *d2[D2_N], *d3[D3_N];
    diag_ptrs(d, d2, d3);
    for (int i = 0; i < D2_N; ++i) a.d2[i] = static_cast<R*>(d2[i]);
    for (int i = 0; i < D3_N; ++i) a.d3[i] = static_cast<R*>(d3[i]);
  }
  a.land = f->land;
  if ((f->qc_bl || f->qcfrac_bl) && !(x->cfg.ml_for_nc_flag || x->cfg.ml_for_bl_nc_flag))
    return fail(TEMPO_HIP_E_ARG, "qc_bl/qcfrac_bl need the cloud-number network (ml_for_bl_nc_flag or ml_for_nc_flag)");
  a.qc_bl = static_cast<const R*>(f->qc_bl);
  a.qcfrac_bl = static_cast<const R*>(f->qcfrac_bl);
  a.nlev = dm->nlev;
  a.ni = dm->ni;
  a.nj = dm->nj;
  a.nz = dm->nz;
  a.ncol = dm->ni * dm->nj;
  a.ldk = dm->ldk;
  a.ldj = dm->ldj;
  a.dldk = dm->dldk;
  a.dldj = dm->dldj;
  a.d2ldj = dm->d2ldj;
  int rc = bind_common(x, a, dt, itimestep, sc);
  if (rc) return rc;
  double* vt = static_cast<double*>(x->last_vt);
  if (sig) {
    if (x->launch[sizeof(R) == 8 ? 1 : 0].order < 0) a.compact = 0;
    a.sig = sig;
    HIP_TRY(launch_step_sig(a, x->launch[sizeof(R) == 8 ? 1 : 0], vt, s));
    return TEMPO_HIP_OK;
  }
  hipEvent_t* ev = nullptr;
  if (x->profile && !sc) {
    for (int i = 0; i < 5; ++i) {
      hipEvent_t e;
      HIP_TRY(hipEventCreate(&e));
      x->events.push_back(e);
    }
    ev = &x->events[x->events.size() - 5];
  }
  HIP_TRY(launch_step(a, x->launch[sizeof(R) == 8 ? 1 : 0], vt, s, ev));
  return TEMPO_HIP_OK;
}

// Tangent-linear step: fields and tangents are interleaved into dual
// arrays (compact layout, column c = i + j*ni), stepped, and split back.
template <class T>
int run_tlm(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_fields* ft, const tempo_hip_diags* d,
            const tempo_hip_diags* dt_, const tempo_hip_dims* dm, double dt, int itimestep, hipStream_t s) {
  using D = Dual<T>;
  if ((f->qc_bl || f->qcfrac_bl) && !(x->cfg.ml_for_nc_flag || x->cfg.ml_for_bl_nc_flag))
    return fail(TEMPO_HIP_E_ARG, "qc_bl/qcfrac_bl need the cloud-number network (ml_for_bl_nc_flag or ml_for_nc_flag)");
  if (x->cfg.refl10cm_from_melting_flag)
    return fail(TEMPO_HIP_E_UNSUPPORTED, "the tangent-linear step does not cover the melting-layer reflectivity");
  const int ncol = dm->ni * dm->nj, nz = dm->nz;
  const size_t n3 = size_t(ncol) * nz;
  const bool bl = f->qc_bl && f->qcfrac_bl;
  HIP_TRY(x->tl_state.ensure((F_NFIELDS + (bl ? 2 : 0)) * n3 * sizeof(D)));
  HIP_TRY(x->tl_diag.ensure((D2_N * size_t(ncol) + D3_N * n3) * sizeof(D)));
  StepArgs<D> a;
  std::memset(&a, 0, sizeof(a));
  void *fp[F_NFIELDS], *tp[F_NFIELDS];
  field_ptrs(f, fp);
  field_ptrs(ft, tp);
  D* st = x->tl_state.as<D>();
  DualGeom g3{dm->ni, dm->nj, nz, dm->ldk, dm->ldj};
  // one launch per layout, in and out
  DualBatch<T> pk{};
  int npk = 0;
  for (int i = 0; i < F_NFIELDS; ++i) {
    if (!fp[i]) continue;
    a.f[i] = st + size_t(i) * n3;
    pk.v[npk] = static_cast<T*>(fp[i]);
    pk.t[npk] = static_cast<T*>(tp[i]);
    pk.d[npk++] = a.f[i];
  }
  const int nstate = npk;
  if (bl) {  // boundary-layer cloud: constants of the step (zero tangent)
    D* qbl = st + F_NFIELDS * n3;
    pk.v[npk] = static_cast<T*>(const_cast<void*>(f->qc_bl));
    pk.d[npk++] = qbl;
    pk.v[npk] = static_cast<T*>(const_cast<void*>(f->qcfrac_bl));
    pk.d[npk++] = qbl + n3;
    a.qc_bl = qbl;
    a.qcfrac_bl = qbl + n3;
  }
  HIP_TRY(launch_dual_pack_n(pk, npk, g3, s));
  void *d2[D2_N] = {}, *d3[D3_N] = {}, *t2[D2_N] = {}, *t3[D3_N] = {};
  if (d) diag_ptrs(d, d2, d3);
  if (dt_) diag_ptrs(dt_, t2, t3);
  D* dg = x->tl_diag.as<D>();
  for (int i = 0; i < D2_N; ++i)
    if (d2[i] || t2[i]) a.d2[i] = dg + size_t(i) * ncol;
  for (int i = 0; i < D3_N; ++i)
    if (d3[i] || t3[i]) a.d3[i] = dg + D2_N * size_t(ncol) + size_t(i) * n3;
  a.land = f->land;
  a.nlev = dm->nlev;
  a.ni = ncol;
  a.nj = 1;
  a.nz = nz;
  a.ncol = ncol;
  a.ldk = ncol;
  a.ldj = (long long)n3;
  a.dldk = ncol;
  a.dldj = (long long)n3;
  a.d2ldj = ncol;
  int rc = bind_common(x, a, dt, itimestep);
  if (rc) return rc;
  HIP_TRY(launch_step_tlm(a, x->launch[sizeof(T) == 8 ? 1 : 0], x->vtbuf.as<Dual<double>>(), s));
  HIP_TRY(launch_dual_unpack_n(pk, nstate, g3, nullptr, s));  // the state's entries come first
  DualGeom g2{dm->ni, dm->nj, 1, 0, dm->d2ldj};
  DualGeom gd3{dm->ni, dm->nj, nz, dm->dldk, dm->dldj};
  DualBatch<T> u2{}, u3{};
  int n2 = 0, nd3 = 0;
  for (int i = 0; i < D2_N; ++i) {
    if (!a.d2[i]) continue;
    u2.v[n2] = static_cast<T*>(d2[i]);
    u2.t[n2] = static_cast<T*>(t2[i]);
    u2.d[n2++] = a.d2[i];
  }
  for (int i = 0; i < D3_N; ++i) {
    if (!a.d3[i]) continue;
    u3.v[nd3] = static_cast<T*>(d3[i]);
    u3.t[nd3] = static_cast<T*>(t3[i]);
    u3.d[nd3++] = a.d3[i];
  }
  HIP_TRY(launch_dual_unpack_n(u2, n2, g2, nullptr, s));
  HIP_TRY(launch_dual_unpack_n(u3, nd3, gd3, dm->nlev, s));
  return TEMPO_HIP_OK;
}

// Adjoint step: tangent passes of the dual step plus S^T (tempo_adjoint.hpp).
template <class T>
int run_adjoint(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_fields* yb, const tempo_hip_diags* db,
                const tempo_hip_fields* xb, const tempo_hip_dims* dm, double dt, int itimestep, hipStream_t s) {
  using D = Dual<T>;
  if (x->cfg.semi_sedi_flag)
    return fail(TEMPO_HIP_E_UNSUPPORTED, "the adjoint covers flux-form sedimentation only");
  if ((f->qc_bl || f->qcfrac_bl) && !(x->cfg.ml_for_nc_flag || x->cfg.ml_for_bl_nc_flag))
    return fail(TEMPO_HIP_E_ARG, "qc_bl/qcfrac_bl need the cloud-number network (ml_for_bl_nc_flag or ml_for_nc_flag)");
  // qc_bl and qcfrac_bl enter only the effective radii, which are not among
  // the adjoint's outputs: they are not bound
  if (x->cfg.refl10cm_from_melting_flag)
    return fail(TEMPO_HIP_E_UNSUPPORTED, "the adjoint does not cover the melting-layer reflectivity");
  if (!f->t) return fail(TEMPO_HIP_E_UNSUPPORTED, "the adjoint takes temperature input t (not th/pii)");
  const int ncol = dm->ni * dm->nj, nz = dm->nz;
  const size_t n3 = size_t(ncol) * nz, sb = F_NFIELDS * n3 * sizeof(D);
  const size_t plane = scratch_plane(size_t(ncol), size_t(nz));
  const size_t nd = (AY_N + AX_N) * n3 + 4 * size_t(ncol) + (10 + AZ_N + AW_N) * plane + (size_t(nz) + 1) / 2 + (n3 + 2) / 2;
  HIP_TRY(x->tl_state.ensure(sb));
  HIP_TRY(x->adj_in.ensure(sb));
  HIP_TRY(x->adj_mem.ensure(nd * sizeof(double)));
  double* mem = x->adj_mem.as<double>();
  AdjArgs g;
  double* ybar = mem;
  g.ybar = ybar;
  g.xbar = ybar + AY_N * n3;
  g.ubar = g.xbar + AX_N * n3;
  g.zbar = g.ubar + 10 * plane;
  double* pbar = g.zbar + AZ_N * plane;
  g.pbar = pbar;
  g.work = pbar + 4 * size_t(ncol);
  g.lvl_on = reinterpret_cast<int*>(g.work + AW_N * plane);
  g.list = reinterpret_cast<unsigned*>(g.work + AW_N * plane + (size_t(nz) + 1) / 2);
  g.count = g.list + n3;

  StepArgs<D> a;
  std::memset(&a, 0, sizeof(a));
  void* fp[F_NFIELDS];
  field_ptrs(f, fp);
  D* in = x->adj_in.as<D>();
  D* st = x->tl_state.as<D>();
  const DualGeom g3{dm->ni, dm->nj, nz, dm->ldk, dm->ldj};
  // the inputs, the output cotangents and the precipitation cotangents, one
  // launch per layout
  DualBatch<T> pk{};
  int npk = 0;
  for (int i = 0; i < F_NFIELDS; ++i) {
    if (!fp[i]) continue;
    pk.v[npk] = static_cast<T*>(fp[i]);
    pk.d[npk++] = in + size_t(i) * n3;
    a.f[i] = st + size_t(i) * n3;
  }
  HIP_TRY(launch_dual_pack_n(pk, npk, g3, s));
  void* yp[F_NFIELDS] = {};
  if (yb) field_ptrs(yb, yp);
  PlaneBatch<T, double> yc{};
  int nyc = 0;
  g.y_on = 0;
  for (int q = 0; q < AY_REFL; ++q) {
    if (!a.f[adj_y_field(q)] || !yp[adj_y_field(q)]) continue;
    g.y_on |= 1u << q;
    yc.src[nyc] = static_cast<const T*>(yp[adj_y_field(q)]);
    yc.dst[nyc++] = ybar + size_t(q) * n3;
  }
  HIP_TRY(launch_to_compact_n(yc, nyc, g3, s));
  void *d2[D2_N] = {}, *d3[D3_N] = {};
  if (db) diag_ptrs(db, d2, d3);
  const DualGeom gd3{dm->ni, dm->nj, nz, dm->dldk, dm->dldj};
  const DualGeom g2{dm->ni, dm->nj, 1, 0, dm->d2ldj};
  if (d3[D3_REFL]) {
    g.y_on |= 1u << AY_REFL;
    PlaneBatch<T, double> rb{};
    rb.src[0] = static_cast<const T*>(d3[D3_REFL]);
    rb.dst[0] = ybar + size_t(AY_REFL) * n3;
    HIP_TRY(launch_to_compact_n(rb, 1, gd3, s));
  }
  const int pmap[4] = {D2_RAIN, D2_GRAUPEL, D2_SNOW, D2_ICE};  // S^T order: rain, graupel, snow, ice
  PlaneBatch<T, double> pc{};
  for (int q = 0; q < 4; ++q) {
    pc.src[q] = static_cast<const T*>(d2[pmap[q]]);
    pc.dst[q] = pbar + size_t(q) * ncol;
  }
  HIP_TRY(launch_to_compact_n(pc, 4, g2, s));
  a.land = f->land;
  a.nlev = dm->nlev;
  a.ni = ncol;
  a.nj = 1;
  a.nz = nz;
  a.ncol = ncol;
  a.ldk = ncol;
  a.ldj = (long long)n3;
  a.dldk = ncol;
  a.dldj = (long long)n3;
  a.d2ldj = ncol;
  int rc = bind_common(x, a, dt, itimestep);
  if (rc) return rc;
  void* xp[F_NFIELDS] = {};
  if (xb) field_ptrs(xb, xp);
  bool have_x[AX_N];
  for (int i = 0; i < AX_N; ++i) have_x[i] = fp[adj_x_field(i)] && xp[adj_x_field(i)];
  // the local passes' scratch: of a large batch the forward's, done with by
  // then; a smaller one's would leave launches that do not fill the chip, so
  // it gets its own, up to kLocalRoom point-directions
  constexpr size_t kLocalRoom = size_t(1) << 21;
  int ndir = 0;
  for (bool h : have_x) ndir += h;
  const bool own_scr = n3 < kLocalRoom && ndir > 0;
  // snapshots: for the lane-per-column sedimentation (nz > 128) the scratch
  // after A, and the post-sedimentation tendency values (10 FP64 planes)
  // where they do not stay in the scratch
  const size_t srb = SR_N * a.plane * sizeof(D), sdb = SD_N * a.plane * sizeof(Dual<double>);
  const bool wave_b = nz <= kSedLevels;
  AdjSnap snap{nullptr, nullptr, nullptr};
  if (!wave_b) {
    HIP_TRY(x->adj_snap.ensure(srb + 2 * sdb));
    char* sp = static_cast<char*>(x->adj_snap.p);
    snap = AdjSnap{sp, sp + srb, sp + srb + sdb};
  } else if (!own_scr) {
    HIP_TRY(x->adj_snap.ensure(10 * a.plane * sizeof(double)));
    snap.sd_b = x->adj_snap.p;
  }
  // out of place: inputs in adj_in, post-check state in tl_state; no pass
  // stores a new state
  for (int i = 0; i < F_NFIELDS; ++i) {
    a.f[i] = fp[i] ? in + size_t(i) * n3 : nullptr;
    a.fa[i] = a.fo[i] = fp[i] ? st + size_t(i) * n3 : nullptr;
  }
  AdjLocal<D> scr{a.sr, a.sd, a.pf, st, a.plane, n3, n3};
  if (own_scr) {
    const size_t m = std::min(kLocalRoom, (n3 * size_t(ndir) + 63) / 64 * 64);
    HIP_TRY(x->adj_local.ensure(m * (SD_N * sizeof(Dual<double>) + (SR_N + F_NFIELDS) * sizeof(D) + sizeof(unsigned))));
    scr.sd = x->adj_local.as<Dual<double>>();
    scr.sr = reinterpret_cast<D*>(scr.sd + SD_N * m);
    scr.fa = scr.sr + SR_N * m;
    scr.pf = reinterpret_cast<unsigned*>(scr.fa + F_NFIELDS * m);
    scr.plane = scr.fplane = scr.room = m;
  }
  HIP_TRY(launch_adjoint(a, g, x->vtbuf.as<Dual<double>>(), srb, sdb, snap, scr, have_x, s));
  PlaneBatch<double, T> xc{};
  int nxc = 0;
  for (int i = 0; i < AX_N; ++i)
    if (have_x[i]) {
      xc.src[nxc] = g.xbar + size_t(i) * n3;
      xc.dst[nxc++] = static_cast<T*>(xp[adj_x_field(i)]);
    }
  HIP_TRY(launch_from_compact_n(xc, nxc, g3, s));
  return TEMPO_HIP_OK;
}

// check_run_args and check_emission_args: an empty batch (ni or nj zero) is
// a no-op, as the reference's loops over an empty tile; the entry points
// return TEMPO_HIP_OK for it without looking at the arrays
constexpr int kEmptyBatch = 1;
int ok_if_empty(int rc) { return rc == kEmptyBatch ? TEMPO_HIP_OK : rc; }

int check_run_args(const tempo_hip_fields* f, const tempo_hip_dims* dm, double dt) {
  if (!f || !dm) return fail(TEMPO_HIP_E_ARG, "NULL fields/dims");
  if (dm->ni < 0 || dm->nj < 0) return fail(TEMPO_HIP_E_ARG, "bad dims (negative ni or nj)");
  if (dm->ni == 0 || dm->nj == 0) return kEmptyBatch;
  if (dm->nz < 2) return fail(TEMPO_HIP_E_ARG, "bad dims (need nz >= 2)");
  if (dm->ldk < dm->ni) return fail(TEMPO_HIP_E_ARG, "ldk smaller than ni");
  if (dm->nj > 1 && dm->ldj < dm->ldk * dm->nz) return fail(TEMPO_HIP_E_ARG, "ldj too small");
  if (!(dt > 0.0)) return fail(TEMPO_HIP_E_ARG, "dt must be positive");
  if (!f->p || !f->w || !f->dz || !f->qv || !f->qc || !f->qr || !f->qi || !f->qs || !f->qg || !f->ni || !f->nr)
    return fail(TEMPO_HIP_E_ARG, "missing required field (p, w, dz, qv, qc, qr, qi, qs, qg, ni, nr)");
  if (!f->t && !(f->th && f->pii)) return fail(TEMPO_HIP_E_ARG, "need t, or th and pii");
  return TEMPO_HIP_OK;
}

// ---- host arrays ---------------------------------------------------------
// A host-array step runs as a pipeline over slabs of columns (ranges of j,
// or of i when nj == 1).  Host threads copy slab s's inputs from the
// caller's (pageable) arrays into pinned memory and the upload stream moves
// them to the device copies; the compute stream steps the slab's columns
// there; the download stream moves the slab's updated fields and
// diagnostics into pinned memory, from which host threads copy them into
// the caller's arrays two slabs later.  Uploads and downloads of different
// slabs overlap (the link is full duplex), the host copies overlap both,
// and each column's step is the device path's.

// Slabs unless set: n slabs cost n times a slab's launches and joins and leave
// 1/n of the transfers at either end of the pipeline without a partner, so
// that the best n grows as the root of the bytes.  Uploads of 36 MB (5,000 x 60
// FP64 fields): 1 slab 2.52 ms, 3 2.12, 6 2.53; 144 MB: 2 6.9, 6 6.0, 12 6.4;
// 432 MB: 4 15.0, 8 13.7, 12 14.1.
constexpr double kSlabRoot = double(size_t(4) << 20);
constexpr int kMaxSlabs = 32;

// elements of one array in one slab: n rows of len elements at element
// offset base + r*pitch of the array (packed row after row in pinned memory)
struct Span {
  size_t base, len, pitch;
  int n;
};

// array kinds: state (ldk, ldj), 3-D diagnostic (dldk, dldj), 2-D
// diagnostic (d2ldj)
enum { K_STATE = 0, K_DIAG3 = 1, K_DIAG2 = 2 };

struct Xfer {
  void* host;
  void* dev;
  int kind;
  bool pinned;  // the caller's array is page-locked: the copy engines move it directly
};

// whether [p, p + bytes) starts and ends in page-locked host memory
bool host_pinned(const void* p, size_t bytes) {
  for (const char* q : {static_cast<const char*>(p), static_cast<const char*>(p) + bytes - 1}) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, q) != hipSuccess) {
      (void)hipGetLastError();  // pageable memory: not an error of the step
      return false;
    }
    if (at.type != hipMemoryTypeHost) return false;
  }
  return true;
}

struct SlabPlan {
  bool along_j;  // slabs of j (whole i rows), else of i (nj == 1)
  int count, width, total;
  int lo(int s) const { return s * width; }
  int hi(int s) const { return std::min(total, (s + 1) * width); }
};

SlabPlan plan_slabs(const tempo_hip_dims* dm, size_t up_bytes, int tuned) {
  SlabPlan p{dm->nj > 1, 1, 0, 0};
  p.total = p.along_j ? dm->nj : dm->ni;
  const int most = p.along_j ? dm->nj : std::max(1, dm->ni / 256);  // i slabs of at least 256 columns
  int n = tuned > 0 ? tuned : int(std::min<double>(kMaxSlabs, std::sqrt(double(up_bytes) / kSlabRoot) + 0.5));
  n = std::max(1, std::min(n, most));
  if (n == 1) p.along_j = true;  // one slab: the arrays' whole spans
  if (p.along_j) p.total = dm->nj;
  p.width = (p.total + n - 1) / n;
  p.count = (p.total + p.width - 1) / p.width;
  return p;
}

Span slab_span(const tempo_hip_dims* dm, const SlabPlan& p, int s, int kind) {
  const size_t lo = size_t(p.lo(s)), m = size_t(p.hi(s)) - lo;
  const size_t ldk = kind == K_STATE ? size_t(dm->ldk) : kind == K_DIAG3 ? size_t(dm->dldk) : 0;
  const size_t ldj = kind == K_STATE ? size_t(dm->ldj) : kind == K_DIAG3 ? size_t(dm->dldj) : size_t(dm->d2ldj);
  const size_t nk = kind == K_DIAG2 ? 1 : size_t(dm->nz);
  if (p.along_j) {
    const size_t len = (m - 1) * ldj + (nk - 1) * ldk + size_t(dm->ni);
    return Span{lo * ldj, len, len, 1};
  }
  if (nk == 1 || ldk == m) return Span{lo, m * nk, m * nk, 1};
  return Span{lo, m, ldk, int(nk)};
}

// the slab's sub-box of an array of the given kind: element offset of its
// first point, and its geometry for the conversion kernels
size_t slab_base(const tempo_hip_dims* dm, const SlabPlan& p, int s, int kind) {
  const size_t lo = size_t(p.lo(s));
  if (!p.along_j) return lo;
  return lo * size_t(kind == K_STATE ? dm->ldj : kind == K_DIAG3 ? dm->dldj : dm->d2ldj);
}
DualGeom slab_geom(const tempo_hip_dims* dm, const SlabPlan& p, int s, int kind) {
  const int m = p.hi(s) - p.lo(s);
  const int ni = p.along_j ? dm->ni : m, nj = p.along_j ? m : 1;
  if (kind == K_STATE) return DualGeom{ni, nj, dm->nz, dm->ldk, dm->ldj};
  if (kind == K_DIAG3) return DualGeom{ni, nj, dm->nz, dm->dldk, dm->dldj};
  return DualGeom{ni, nj, 1, 0, dm->d2ldj};
}

int ensure_host_staging(tempo_hip_ctx* x, unsigned threads) {
  for (hipStream_t* st : {&x->host_stream, &x->up_stream, &x->down_stream}) {
    if (!*st) HIP_TRY(hipStreamCreateWithFlags(st, hipStreamNonBlocking));
    HIP_TRY(hipStreamSynchronize(*st));  // nothing of an earlier call still uses the pinned buffers
  }
  for (hipEvent_t& e : x->ev_up)
    if (!e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  for (hipEvent_t& e : x->ev_dn)
    if (!e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (!x->ev_step) HIP_TRY(hipEventCreateWithFlags(&x->ev_step, hipEventDisableTiming));
  if (!x->pool || x->pool->threads() != threads) x->pool.reset(new CopyPool(threads));
  return TEMPO_HIP_OK;
}

// n pinned buffers of at least `need` bytes each (grown in 16 MB steps)
int ensure_pinned(void** b, int n, size_t& have, size_t need) {
  if (need <= have) return TEMPO_HIP_OK;
  need = (need + (size_t(16) << 20) - 1) / (size_t(16) << 20) * (size_t(16) << 20);
  for (int i = 0; i < n; ++i) {
    if (b[i]) HIP_TRY(hipHostFree(b[i]));
    b[i] = nullptr;
  }
  have = 0;
  for (int i = 0; i < n; ++i) HIP_TRY(hipHostMalloc(&b[i], need, hipHostMallocDefault));
  have = need;
  return TEMPO_HIP_OK;
}

// bytes of the transfers' spans in slab s
size_t slab_bytes(const tempo_hip_dims* dm, const SlabPlan& p, int s, const std::vector<Xfer>& xs) {
  size_t n = 0;
  for (const Xfer& t : xs) {
    if (t.pinned) continue;
    const Span sp = slab_span(dm, p, s, t.kind);
    n += sp.len * size_t(sp.n) * sizeof(double);
  }
  return n;
}

// host copies between the caller's arrays and a slab's pinned buffer
void slab_host_copy(tempo_hip_ctx* x, const tempo_hip_dims* dm, const SlabPlan& p, int s,
                    const std::vector<Xfer>& xs, char* pin, bool to_pinned, std::vector<Piece>& pieces) {
  pieces.clear();
  size_t off = 0;
  for (const Xfer& t : xs) {
    if (t.pinned) continue;
    const Span sp = slab_span(dm, p, s, t.kind);
    char* h = static_cast<char*>(t.host);
    for (int r = 0; r < sp.n; ++r) {
      char* a = h + (sp.base + size_t(r) * sp.pitch) * sizeof(double);
      const size_t n = sp.len * sizeof(double);
      pieces.push_back(to_pinned ? Piece{pin + off, a, n} : Piece{a, pin + off, n});
      off += n;
    }
  }
  x->pool->run(pieces);
}

// copy-engine moves between the device copies and a slab's pinned buffer,
// or the caller's array itself where that is page-locked
int slab_dma(const tempo_hip_dims* dm, const SlabPlan& p, int s, const std::vector<Xfer>& xs, char* pin, bool up,
             hipStream_t st) {
  size_t off = 0;
  for (const Xfer& t : xs) {
    const Span sp = slab_span(dm, p, s, t.kind);
    char* dv = static_cast<char*>(t.dev) + sp.base * sizeof(double);
    char* hv = t.pinned ? static_cast<char*>(t.host) + sp.base * sizeof(double) : pin + off;
    const size_t w = sp.len * sizeof(double), dpitch = sp.pitch * sizeof(double), hpitch = t.pinned ? dpitch : w;
    if (sp.n == 1) {
      HIP_TRY(up ? hipMemcpyAsync(dv, hv, w, hipMemcpyHostToDevice, st)
                 : hipMemcpyAsync(hv, dv, w, hipMemcpyDeviceToHost, st));
    } else {
      HIP_TRY(up ? hipMemcpy2DAsync(dv, dpitch, hv, hpitch, w, size_t(sp.n), hipMemcpyHostToDevice, st)
                 : hipMemcpy2DAsync(hv, hpitch, dv, dpitch, w, size_t(sp.n), hipMemcpyDeviceToHost, st));
    }
    if (!t.pinned) off += w * size_t(sp.n);
  }
  return TEMPO_HIP_OK;
}

// element conversion over the points of a tile (the points a step writes:
// i < ni, k < nk and, with nlev, k < nlev[i + j*ni])
template <class S, class D>
__global__ void __launch_bounds__(256) k_cast_tile(const S* __restrict__ in, D* __restrict__ out, DualGeom g,
                                                   const int* __restrict__ nlev) {
  const int i = int(blockIdx.x) * 256 + int(threadIdx.x), k = int(blockIdx.y), j = int(blockIdx.z);
  if (i >= g.ni) return;
  if (nlev && k >= nlev[i + j * g.ni]) return;
  const size_t e = size_t(i) + size_t(k) * size_t(g.ldk) + size_t(j) * size_t(g.ldj);
  out[e] = D(in[e]);
}
template <class S, class D>
hipError_t cast_tile(const S* in, D* out, const DualGeom& g, const int* nlev, hipStream_t s) {
  hipLaunchKernelGGL((k_cast_tile<S, D>), dim3(unsigned((g.ni + 255) / 256), unsigned(g.nk), unsigned(g.nj)), dim3(256),
                     0, s, in, out, g, nlev);
  return hipGetLastError();
}

// tempo_hip_run_host(_prec): the caller's FP64 host arrays are copied to the
// device (the diagnostics only where the step does not write every point of
// their spans: padded rows, or ragged columns), stepped in `precision` (FP32:
// on FP32 copies, converted back at the points the step writes) and the
// updated fields and diagnostics copied back, slab by slab.
int run_host_impl(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_diags* d, const tempo_hip_dims* dm,
                  double dt, int itimestep, int precision) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_run_args(f, dm, dt);
  if (rc) return ok_if_empty(rc);
  const bool fp32 = precision == TEMPO_HIP_FP32;
  const LaunchCfg& lc = x->launch[fp32 ? 0 : 1];
  if ((rc = ensure_host_staging(x, unsigned(lc.host_threads)))) return rc;
  hipStream_t cs = x->host_stream;
  const size_t n3 = size_t(dm->ldj) * (dm->nj - 1) + size_t(dm->ldk) * (dm->nz - 1) + dm->ni;
  const size_t nd3 = size_t(dm->dldj) * (dm->nj - 1) + size_t(dm->dldk) * (dm->nz - 1) + dm->ni;
  const size_t nd2 = size_t(dm->d2ldj) * (dm->nj - 1) + dm->ni;
  constexpr int kNf = 21;  // the 19 fields, qc_bl, qcfrac_bl
  void* const hf[kNf] = {f->t,  f->th, f->pii, f->p,  f->w,  f->dz,   f->qv,   f->qc, f->qr,   f->qi,    f->qs,
                         f->qg, f->ni, f->nr,  f->nc, f->nwfa, f->nifa, f->ng, f->qb, const_cast<void*>(f->qc_bl),
                         const_cast<void*>(f->qcfrac_bl)};
  // fields the step writes: temperature (t, else th) and the water species,
  // numbers and aerosols
  auto written = [&](int i) { return i == 0 || (i == 1 && !f->t) || (i >= 6 && i <= 18); };
  const int nd = sizeof(tempo_hip_diags) / sizeof(void*);
  void** hd = reinterpret_cast<void**>(const_cast<tempo_hip_diags*>(d));
  if (d) {
    bool has3 = false, has2 = false;
    for (int i = 0; i < nd; ++i)
      if (hd[i]) (i < D2_N ? has2 : has3) = true;
    if (has3 && (dm->dldk < dm->ni || (dm->nj > 1 && dm->dldj < dm->dldk * dm->nz)))
      return fail(TEMPO_HIP_E_ARG, "3-D diagnostic strides overlap (need dldk >= ni, dldj >= dldk*nz)");
    if (has2 && dm->nj > 1 && dm->d2ldj < dm->ni)
      return fail(TEMPO_HIP_E_ARG, "2-D diagnostic stride overlaps (need d2ldj >= ni)");
  }
  if (x->stage.size() < size_t(kNf + nd)) x->stage.resize(kNf + nd);
  if (fp32 && x->stage32.size() < size_t(kNf + nd)) x->stage32.resize(kNf + nd);
  std::vector<Xfer> up, down;
  for (int i = 0; i < kNf; ++i) {
    if (!hf[i]) continue;
    HIP_TRY(x->stage[i].ensure(n3 * sizeof(double)));
    const bool pin = host_pinned(hf[i], n3 * sizeof(double));
    up.push_back({hf[i], x->stage[i].p, K_STATE, pin});
    if (written(i)) down.push_back({hf[i], x->stage[i].p, K_STATE, pin});
    if (fp32) HIP_TRY(x->stage32[i].ensure(n3 * sizeof(float)));
  }
  // diagnostics: uploaded where the step leaves points of their spans
  // unwritten (padding between rows, levels k >= nlev[c]), so that those
  // come back unchanged
  const bool dense3 = !dm->nlev && dm->dldk == dm->ni && (dm->nj == 1 || dm->dldj == dm->dldk * dm->nz);
  const bool dense2 = dm->nj == 1 || dm->d2ldj == dm->ni;
  for (int i = 0; d && i < nd; ++i) {
    if (!hd[i]) continue;
    const bool two = i < D2_N;
    const size_t n = two ? nd2 : nd3;
    HIP_TRY(x->stage[kNf + i].ensure(n * sizeof(double)));
    const bool pin = host_pinned(hd[i], n * sizeof(double));
    if (!(two ? dense2 : dense3)) up.push_back({hd[i], x->stage[kNf + i].p, two ? K_DIAG2 : K_DIAG3, pin});
    down.push_back({hd[i], x->stage[kNf + i].p, two ? K_DIAG2 : K_DIAG3, pin});
    if (fp32) HIP_TRY(x->stage32[kNf + i].ensure(n * sizeof(float)));
  }
  const int ncol = dm->ni * dm->nj;
  const int* land = nullptr;
  const int* nlev = nullptr;
  if (f->land) {
    HIP_TRY(x->stage_land.ensure(ncol * sizeof(int)));
    HIP_TRY(hipMemcpyAsync(x->stage_land.p, f->land, ncol * sizeof(int), hipMemcpyHostToDevice, cs));
    land = x->stage_land.as<int>();
  }
  if (dm->nlev) {
    HIP_TRY(x->stage_nlev.ensure(ncol * sizeof(int)));
    HIP_TRY(hipMemcpyAsync(x->stage_nlev.p, dm->nlev, ncol * sizeof(int), hipMemcpyHostToDevice, cs));
    nlev = x->stage_nlev.as<int>();
  }
  HIP_TRY(hipStreamSynchronize(cs));  // land and nlev are pageable: their copies finish before the caller's return

  size_t up_total = 0;  // all uploads, pinned or not: the slabs also pipeline the copy engines' moves
  for (const Xfer& t : up) up_total += (t.kind == K_STATE ? n3 : t.kind == K_DIAG3 ? nd3 : nd2) * sizeof(double);
  const SlabPlan plan = plan_slabs(dm, up_total, lc.host_slabs);
  // slab 0 is the widest
  if ((rc = ensure_pinned(x->pin_up, 2, x->pin_up_bytes, slab_bytes(dm, plan, 0, up)))) return rc;
  if ((rc = ensure_pinned(x->pin_dn, 3, x->pin_dn_bytes, slab_bytes(dm, plan, 0, down)))) return rc;

  // the step of slab s on the compute stream, on the device copies
  auto step = [&](int s) -> int {
    const int lo = plan.lo(s), m = plan.hi(s) - lo;
    const size_t col0 = plan.along_j ? size_t(lo) * dm->ni : size_t(lo);
    const size_t b3 = slab_base(dm, plan, s, K_STATE), bd3 = slab_base(dm, plan, s, K_DIAG3),
                 bd2 = slab_base(dm, plan, s, K_DIAG2);
    const DualGeom g3 = slab_geom(dm, plan, s, K_STATE), gd3 = slab_geom(dm, plan, s, K_DIAG3),
                   gd2 = slab_geom(dm, plan, s, K_DIAG2);
    const int* nl = nlev ? nlev + col0 : nullptr;
    tempo_hip_fields df = *f;
    void** dfp[kNf] = {&df.t,  &df.th, &df.pii, &df.p,  &df.w,  &df.dz,   &df.qv,   &df.qc, &df.qr,    &df.qi,    &df.qs,
                       &df.qg, &df.ni, &df.nr,  &df.nc, &df.nwfa, &df.nifa, &df.ng, &df.qb,
                       const_cast<void**>(&df.qc_bl), const_cast<void**>(&df.qcfrac_bl)};
    for (int i = 0; i < kNf; ++i) {
      if (!hf[i]) continue;
      double* s64 = x->stage[i].as<double>() + b3;
      if (fp32) {
        float* s32 = x->stage32[i].as<float>() + b3;
        HIP_TRY(cast_tile(s64, s32, g3, nullptr, cs));
        *dfp[i] = s32;
      } else {
        *dfp[i] = s64;
      }
    }
    df.land = land ? land + col0 : nullptr;
    tempo_hip_diags dd{};
    void** ddp = reinterpret_cast<void**>(&dd);
    for (int i = 0; d && i < nd; ++i) {
      if (!hd[i]) continue;
      const bool two = i < D2_N;
      double* s64 = x->stage[kNf + i].as<double>() + (two ? bd2 : bd3);
      if (fp32) {
        float* s32 = x->stage32[kNf + i].as<float>() + (two ? bd2 : bd3);
        if (!(two ? dense2 : dense3)) HIP_TRY(cast_tile(s64, s32, two ? gd2 : gd3, nullptr, cs));
        ddp[i] = s32;
      } else {
        ddp[i] = s64;
      }
    }
    tempo_hip_dims dms = *dm;
    (plan.along_j ? dms.nj : dms.ni) = m;
    dms.nlev = nl;
    int r = fp32 ? run_impl<float>(x, &df, d ? &dd : nullptr, &dms, dt, itimestep, cs)
                 : run_impl<double>(x, &df, d ? &dd : nullptr, &dms, dt, itimestep, cs);
    if (r || !fp32) return r;
    for (int i = 0; i < kNf; ++i)
      if (hf[i] && written(i))
        HIP_TRY(cast_tile(x->stage32[i].as<float>() + b3, x->stage[i].as<double>() + b3, g3, nl, cs));
    for (int i = 0; d && i < nd; ++i)
      if (hd[i]) {
        const bool two = i < D2_N;
        const size_t b = two ? bd2 : bd3;
        HIP_TRY(cast_tile(x->stage32[kNf + i].as<float>() + b, x->stage[kNf + i].as<double>() + b, two ? gd2 : gd3,
                          two ? nullptr : nl, cs));
      }
    return TEMPO_HIP_OK;
  };

  std::vector<Piece> pieces;
  for (int s = 0; s < plan.count + 2; ++s) {
    if (s < plan.count) {
      const int b = s & 1;
      char* pu = static_cast<char*>(x->pin_up[b]);
      char* pd = static_cast<char*>(x->pin_dn[s % 3]);
      if (s >= 2) HIP_TRY(hipEventSynchronize(x->ev_up[b]));  // slab s-2's upload has left this buffer
      slab_host_copy(x, dm, plan, s, up, pu, true, pieces);
      if ((rc = slab_dma(dm, plan, s, up, pu, true, x->up_stream))) return rc;
      HIP_TRY(hipEventRecord(x->ev_up[b], x->up_stream));
      HIP_TRY(hipStreamWaitEvent(cs, x->ev_up[b], 0));
      if ((rc = step(s))) return rc;
      HIP_TRY(hipEventRecord(x->ev_step, cs));
      // the host copied slab s-3 out of this buffer in the previous round
      HIP_TRY(hipStreamWaitEvent(x->down_stream, x->ev_step, 0));
      if ((rc = slab_dma(dm, plan, s, down, pd, false, x->down_stream))) return rc;
      HIP_TRY(hipEventRecord(x->ev_dn[s % 3], x->down_stream));
    }
    if (s >= 2) {
      const int o = s - 2;
      HIP_TRY(hipEventSynchronize(x->ev_dn[o % 3]));
      slab_host_copy(x, dm, plan, o, down, static_cast<char*>(x->pin_dn[o % 3]), false, pieces);
    }
  }
  if (plan.count > 1) {  // the scratch holds the last slab's record only
    x->last_ncol = 0;
    x->last_ksub = nullptr;
  }
  return TEMPO_HIP_OK;
}

}  // namespace

extern "C" {

int tempo_hip_init(const tempo_hip_cfg* cfg, const char* table_dir, const char* ccn_path, tempo_hip_ctx** out) {
  if (!cfg || !out) return fail(TEMPO_HIP_E_ARG, "tempo_hip_init: NULL argument");
  *out = nullptr;
  auto* x = new tempo_hip_ctx();
  x->cfg = *cfg;
  int rc;
  auto bail = [&](int r) {
    delete x;
    return r;
  };
  if (hipGetDevice(&x->device) != hipSuccess) return bail(fail(TEMPO_HIP_E_HIP, "no HIP device"));
  HostBins hb;
  build_const(x->cd, hb, cfg->hailaware_flag != 0);
  narrow(x->cd, x->cf);
  {
    std::vector<Const<double>> vd(1, x->cd);
    std::vector<Const<float>> vf(1, x->cf);
    if (upload(x->cd_dev, vd) != hipSuccess || upload(x->cf_dev, vf) != hipSuccess)
      return bail(fail(TEMPO_HIP_E_HIP, "constant upload failed"));
    std::vector<Radar> vr(1);
    build_radar(x->cd, vr[0]);
    if (upload(x->radar, vr) != hipSuccess) return bail(fail(TEMPO_HIP_E_HIP, "constant upload failed"));
  }
  if ((rc = upload_small_tables(x))) return bail(rc);
  std::string ccn = ccn_path ? ccn_path : (table_dir ? std::string(table_dir) + "/ccn_activate.bin" : "");
  if (ccn.empty()) return bail(fail(TEMPO_HIP_E_ARG, "no CCN table path"));
  if ((rc = read_ccn(x, ccn))) return bail(rc);
  if (table_dir) {
    if ((rc = read_tables(x, table_dir))) return bail(rc);
  } else {
    if ((rc = build_tables_gpu(x))) return bail(rc);
  }
  if ((rc = pack_tables(x))) return bail(rc);
  *out = x;
  return TEMPO_HIP_OK;
}

int tempo_hip_reserve(tempo_hip_ctx* x, int ncol, int nz) {
  if (!x || ncol <= 0 || nz <= 0) return fail(TEMPO_HIP_E_ARG, "tempo_hip_reserve: bad arguments");
  return ensure_scratch(x, size_t(ncol), size_t(nz));
}

int tempo_hip_run(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_diags* d, const tempo_hip_dims* dm,
                  double dt, int itimestep, int precision, void* stream) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_run_args(f, dm, dt);
  if (rc) return ok_if_empty(rc);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (precision == TEMPO_HIP_FP32) return run_impl<float>(x, f, d, dm, dt, itimestep, s);
  if (precision == TEMPO_HIP_FP64) return run_impl<double>(x, f, d, dm, dt, itimestep, s);
  return fail(TEMPO_HIP_E_ARG, "precision must be TEMPO_HIP_FP32 or TEMPO_HIP_FP64");
}

int tempo_hip_branch_signature(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_diags* d,
                               const tempo_hip_dims* dm, double dt, int itimestep, int precision, unsigned* sig,
                               void* stream) {
  if (!x || !sig) return fail(TEMPO_HIP_E_ARG, "NULL context or signature array");
  int rc = check_run_args(f, dm, dt);
  if (rc) return ok_if_empty(rc);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (precision == TEMPO_HIP_FP32) return run_impl<float>(x, f, d, dm, dt, itimestep, s, sig);
  if (precision == TEMPO_HIP_FP64) return run_impl<double>(x, f, d, dm, dt, itimestep, s, sig);
  return fail(TEMPO_HIP_E_ARG, "precision must be TEMPO_HIP_FP32 or TEMPO_HIP_FP64");
}

static int check_emission_args(const void* nwfa, const void* nwfa2d, const tempo_hip_dims* dm, int k) {
  if (!dm) return fail(TEMPO_HIP_E_ARG, "NULL dims");
  if (dm->ni < 0 || dm->nj < 0) return fail(TEMPO_HIP_E_ARG, "bad dims (negative ni or nj)");
  if (dm->ni == 0 || dm->nj == 0) return kEmptyBatch;
  if (!nwfa || !nwfa2d) return fail(TEMPO_HIP_E_ARG, "NULL nwfa or nwfa2d");
  if (dm->nz <= 0 || k < 0 || k >= dm->nz)
    return fail(TEMPO_HIP_E_ARG, "bad dims or level (need 0 <= k < nz)");
  if (dm->ldk < dm->ni || (dm->nj > 1 && (dm->ldj < dm->ldk * dm->nz || dm->d2ldj < dm->ni)))
    return fail(TEMPO_HIP_E_ARG, "leading dimensions too small");
  return TEMPO_HIP_OK;
}

int tempo_hip_aerosol_surface_emissions(tempo_hip_ctx* x, double dt, void* nwfa, const void* nwfa2d,
                                        const tempo_hip_dims* dm, int k, int precision, void* stream) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_emission_args(nwfa, nwfa2d, dm, k);
  if (rc) return ok_if_empty(rc);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (precision == TEMPO_HIP_FP32)
    HIP_TRY(launch_surface_emissions(static_cast<float*>(nwfa), static_cast<const float*>(nwfa2d), dm->ni, dm->nj,
                                     dm->ldk, dm->ldj, dm->d2ldj, k, dt, s));
  else if (precision == TEMPO_HIP_FP64)
    HIP_TRY(launch_surface_emissions(static_cast<double*>(nwfa), static_cast<const double*>(nwfa2d), dm->ni, dm->nj,
                                     dm->ldk, dm->ldj, dm->d2ldj, k, dt, s));
  else
    return fail(TEMPO_HIP_E_ARG, "bad precision");
  return TEMPO_HIP_OK;
}

}  // extern "C"

namespace {

// the public check routines: which = 0 cloud, 1 ice, 2 snow; p holds rho,
// q, nn, ncsave, r, num, qten, nten, ilam, mvd (working precision)
struct CheckPtrs {
  const void* rho;
  int* l;
  void *q, *nn;
  const void* ncsave;
  void *r, *num, *qten, *nten, *ilam, *mvd;
};

int check_ptrs_ok(int which, int n, const CheckPtrs& p, double dt) {
  if (n < 0 || !(dt > 0.0)) return fail(TEMPO_HIP_E_ARG, "check_and_update: bad n or dt");
  bool ok = p.rho && p.l && p.q && p.r && p.qten;
  if (which == 0) ok = ok && p.num && p.nten && p.ilam && p.mvd;
  if (which == 1) ok = ok && p.nn && p.num && p.nten && p.ilam;
  return ok ? TEMPO_HIP_OK : fail(TEMPO_HIP_E_ARG, "check_and_update: NULL array");
}

template <class R>
int run_check(tempo_hip_ctx* x, int which, int n, const CheckPtrs& p, double dt, hipStream_t s) {
  CheckArgs<R> g;
  g.n = n;
  g.dt = R(dt);
  g.odt = sizeof(R) == 4 ? R(1.0f / float(dt)) : R(1.0 / dt);
  g.rho = static_cast<const R*>(p.rho);
  g.l = p.l;
  g.q = static_cast<R*>(p.q);
  g.nn = static_cast<R*>(p.nn);
  g.ncsave = static_cast<const R*>(p.ncsave);
  g.r = static_cast<R*>(p.r);
  g.num = static_cast<R*>(p.num);
  g.qten = static_cast<R*>(p.qten);
  g.nten = static_cast<R*>(p.nten);
  g.ilam = static_cast<R*>(p.ilam);
  g.mvd = static_cast<R*>(p.mvd);
  g.cst = static_cast<const Const<R>*>(sizeof(R) == 8 ? x->cd_dev.p : x->cf_dev.p);
  HIP_TRY(launch_check_update(g, which, s));
  return TEMPO_HIP_OK;
}

int check_device(tempo_hip_ctx* x, int which, int n, const CheckPtrs& p, double dt, int precision, void* stream) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_ptrs_ok(which, n, p, dt);
  if (rc) return rc;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (precision == TEMPO_HIP_FP32) return run_check<float>(x, which, n, p, dt, s);
  if (precision == TEMPO_HIP_FP64) return run_check<double>(x, which, n, p, dt, s);
  return fail(TEMPO_HIP_E_ARG, "precision must be TEMPO_HIP_FP32 or TEMPO_HIP_FP64");
}

// host arrays: every given array staged through device memory and back
int check_host(tempo_hip_ctx* x, int which, int n, const CheckPtrs& p, double dt) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_ptrs_ok(which, n, p, dt);
  if (rc || n == 0) return rc;
  const void* host[11] = {p.rho, p.l, p.q, p.nn, p.ncsave, p.r, p.num, p.qten, p.nten, p.ilam, p.mvd};
  void* dev[11] = {};
  if (x->stage.size() < 11) x->stage.resize(11);
  for (int i = 0; i < 11; ++i) {
    if (!host[i]) continue;
    const size_t b = size_t(n) * (i == 1 ? sizeof(int) : sizeof(double));
    HIP_TRY(x->stage[i].ensure(b));
    HIP_TRY(hipMemcpy(x->stage[i].p, host[i], b, hipMemcpyHostToDevice));
    dev[i] = x->stage[i].p;
  }
  CheckPtrs d{dev[0], static_cast<int*>(dev[1]), dev[2], dev[3], dev[4], dev[5], dev[6], dev[7], dev[8], dev[9], dev[10]};
  if ((rc = run_check<double>(x, which, n, d, dt, nullptr))) return rc;
  HIP_TRY(hipDeviceSynchronize());
  for (int i = 1; i < 11; ++i) {
    if (!host[i] || i == 4) continue;  // rho and ncsave are inputs only
    const size_t b = size_t(n) * (i == 1 ? sizeof(int) : sizeof(double));
    HIP_TRY(hipMemcpy(const_cast<void*>(host[i]), dev[i], b, hipMemcpyDeviceToHost));
  }
  return TEMPO_HIP_OK;
}

}  // namespace

extern "C" {

int tempo_hip_cloud_check_and_update(tempo_hip_ctx* x, int n, const void* rho, int* l_qc, void* qc1d, void* nc1d,
                                     const void* ncsave, void* rc, void* nc, void* qcten, void* ncten, void* ilamc,
                                     void* mvd_c, double dt, int precision, void* stream) {
  return check_device(x, 0, n, CheckPtrs{rho, l_qc, qc1d, nc1d, ncsave, rc, nc, qcten, ncten, ilamc, mvd_c}, dt,
                      precision, stream);
}
int tempo_hip_ice_check_and_update(tempo_hip_ctx* x, int n, const void* rho, int* l_qi, void* qi1d, void* ni1d,
                                   void* ri, void* ni, void* qiten, void* niten, void* ilami, double dt, int precision,
                                   void* stream) {
  return check_device(x, 1, n, CheckPtrs{rho, l_qi, qi1d, ni1d, nullptr, ri, ni, qiten, niten, ilami, nullptr}, dt,
                      precision, stream);
}
int tempo_hip_snow_check_and_update(tempo_hip_ctx* x, int n, const void* rho, int* l_qs, void* qs1d, void* rs,
                                    void* qsten, double dt, int precision, void* stream) {
  return check_device(x, 2, n, CheckPtrs{rho, l_qs, qs1d, nullptr, nullptr, rs, nullptr, qsten, nullptr, nullptr, nullptr},
                      dt, precision, stream);
}
int tempo_hip_cloud_check_and_update_host(tempo_hip_ctx* x, int n, const double* rho, int* l_qc, double* qc1d,
                                          double* nc1d, const double* ncsave, double* rc, double* nc, double* qcten,
                                          double* ncten, double* ilamc, double* mvd_c, double dt) {
  return check_host(x, 0, n, CheckPtrs{rho, l_qc, qc1d, nc1d, ncsave, rc, nc, qcten, ncten, ilamc, mvd_c}, dt);
}
int tempo_hip_ice_check_and_update_host(tempo_hip_ctx* x, int n, const double* rho, int* l_qi, double* qi1d,
                                        double* ni1d, double* ri, double* ni, double* qiten, double* niten,
                                        double* ilami, double dt) {
  return check_host(x, 1, n, CheckPtrs{rho, l_qi, qi1d, ni1d, nullptr, ri, ni, qiten, niten, ilami, nullptr}, dt);
}
int tempo_hip_snow_check_and_update_host(tempo_hip_ctx* x, int n, const double* rho, int* l_qs, double* qs1d,
                                         double* rs, double* qsten, double dt) {
  return check_host(x, 2, n, CheckPtrs{rho, l_qs, qs1d, nullptr, nullptr, rs, nullptr, qsten, nullptr, nullptr, nullptr},
                    dt);
}

int tempo_hip_aerosol_surface_emissions_host(tempo_hip_ctx* x, double dt, double* nwfa, const double* nwfa2d,
                                             const tempo_hip_dims* dm, int k) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_emission_args(nwfa, nwfa2d, dm, k);
  if (rc) return ok_if_empty(rc);
  const size_t n3 = size_t(dm->ldj) * (dm->nj - 1) + size_t(dm->ldk) * (dm->nz - 1) + dm->ni;
  const size_t n2 = size_t(dm->d2ldj) * (dm->nj - 1) + dm->ni;
  if (x->stage.size() < 2) x->stage.resize(2);
  HIP_TRY(x->stage[0].ensure(n3 * sizeof(double)));
  HIP_TRY(x->stage[1].ensure(n2 * sizeof(double)));
  HIP_TRY(hipMemcpy(x->stage[0].p, nwfa, n3 * sizeof(double), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(x->stage[1].p, nwfa2d, n2 * sizeof(double), hipMemcpyHostToDevice));
  HIP_TRY(launch_surface_emissions(x->stage[0].as<double>(), x->stage[1].as<double>(), dm->ni, dm->nj, dm->ldk,
                                   dm->ldj, dm->d2ldj, k, dt, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(nwfa, x->stage[0].p, n3 * sizeof(double), hipMemcpyDeviceToHost));
  return TEMPO_HIP_OK;
}

int tempo_hip_run_host(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_diags* d,
                       const tempo_hip_dims* dm, double dt, int itimestep) {
  return run_host_impl(x, f, d, dm, dt, itimestep, TEMPO_HIP_FP64);
}

int tempo_hip_run_host_prec(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_diags* d,
                            const tempo_hip_dims* dm, double dt, int itimestep, int precision) {
  if (precision != TEMPO_HIP_FP32 && precision != TEMPO_HIP_FP64)
    return fail(TEMPO_HIP_E_ARG, "precision must be TEMPO_HIP_FP32 or TEMPO_HIP_FP64");
  return run_host_impl(x, f, d, dm, dt, itimestep, precision);
}

int tempo_hip_host_alloc(size_t bytes, void** ptr) {
  if (!ptr) return fail(TEMPO_HIP_E_ARG, "NULL pointer argument");
  *ptr = nullptr;
  if (bytes == 0) return fail(TEMPO_HIP_E_ARG, "zero bytes");
  HIP_TRY(hipHostMalloc(ptr, bytes, hipHostMallocDefault));
  return TEMPO_HIP_OK;
}

int tempo_hip_host_free(void* ptr) {
  if (ptr) HIP_TRY(hipHostFree(ptr));
  return TEMPO_HIP_OK;
}

int tempo_hip_table_export(tempo_hip_ctx* x, int table, double* out, size_t n) {
  if (!x || !out) return fail(TEMPO_HIP_E_ARG, "NULL argument");
  const DevBuf* b = nullptr;
  size_t want = 0;
  switch (table) {
    case TEMPO_HIP_TABLE_QR_ACR_QG: b = &x->qg_ref; want = kNQgArr * kNQg1; break;
    case TEMPO_HIP_TABLE_QR_ACR_QS: b = &x->qs_ref; want = kNQsArr * kNQs1; break;
    case TEMPO_HIP_TABLE_FREEZEWATER: b = &x->fz_ref; want = kNFzRArr * kNFzR1 + kNFzCArr * kNFzC1; break;
    default: return fail(TEMPO_HIP_E_ARG, "unknown table id");
  }
  if (n != want) return fail(TEMPO_HIP_E_ARG, "table size mismatch: expected " + std::to_string(want));
  HIP_TRY(hipMemcpy(out, b->p, n * sizeof(double), hipMemcpyDeviceToHost));
  return TEMPO_HIP_OK;
}

int tempo_hip_table_write(tempo_hip_ctx* x, const char* dir) {
  if (!x || !dir) return fail(TEMPO_HIP_E_ARG, "NULL argument");
  struct Item {
    const char* name;
    int id;
    size_t n;
  } items[3] = {{"freeze_water_data_tempo_v3", TEMPO_HIP_TABLE_FREEZEWATER, kNFzRArr * kNFzR1 + kNFzCArr * kNFzC1},
                {"qr_acr_qs_data_tempo_v3", TEMPO_HIP_TABLE_QR_ACR_QS, kNQsArr * kNQs1},
                {"qr_acr_qg_data_tempo_v3", TEMPO_HIP_TABLE_QR_ACR_QG, kNQgArr * kNQg1}};
  for (auto& it : items) {
    std::vector<double> v(it.n);
    int rc = tempo_hip_table_export(x, it.id, v.data(), it.n);
    if (rc) return rc;
    for (auto& e : v) e = bswap(e);
    std::string path = std::string(dir) + "/" + it.name;
    FILE* fp = std::fopen(path.c_str(), "wb");
    if (!fp) return fail(TEMPO_HIP_E_TABLE, "cannot write " + path);
    size_t w = std::fwrite(v.data(), sizeof(double), it.n, fp);
    std::fclose(fp);
    if (w != it.n) return fail(TEMPO_HIP_E_TABLE, "short write " + path);
  }
  return TEMPO_HIP_OK;
}

int tempo_hip_tlm(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_fields* f_tl, const tempo_hip_diags* d,
                  const tempo_hip_diags* d_tl, const tempo_hip_dims* dm, double dt, int itimestep, int precision,
                  void* stream) {
  if (!x || !f_tl) return fail(TEMPO_HIP_E_ARG, "NULL context or tangent fields");
  int rc = check_run_args(f, dm, dt);
  if (rc) return ok_if_empty(rc);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (precision == TEMPO_HIP_FP32) return run_tlm<float>(x, f, f_tl, d, d_tl, dm, dt, itimestep, s);
  if (precision == TEMPO_HIP_FP64) return run_tlm<double>(x, f, f_tl, d, d_tl, dm, dt, itimestep, s);
  return fail(TEMPO_HIP_E_ARG, "precision must be TEMPO_HIP_FP32 or TEMPO_HIP_FP64");
}

int tempo_hip_adjoint(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_fields* ybar,
                      const tempo_hip_diags* dbar, const tempo_hip_fields* xbar, const tempo_hip_dims* dm, double dt,
                      int itimestep, int precision, void* stream) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_run_args(f, dm, dt);
  if (rc) return ok_if_empty(rc);
  if (!x->cfg.refl10cm_flag && dbar && dbar->refl10cm)
    return fail(TEMPO_HIP_E_ARG, "reflectivity cotangent given but refl10cm_flag is off");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (precision == TEMPO_HIP_FP32) return run_adjoint<float>(x, f, ybar, dbar, xbar, dm, dt, itimestep, s);
  if (precision == TEMPO_HIP_FP64) return run_adjoint<double>(x, f, ybar, dbar, xbar, dm, dt, itimestep, s);
  return fail(TEMPO_HIP_E_ARG, "precision must be TEMPO_HIP_FP32 or TEMPO_HIP_FP64");
}

int tempo_hip_tune(tempo_hip_ctx* x, int precision, int key, int value) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  if (precision != TEMPO_HIP_FP32 && precision != TEMPO_HIP_FP64) return fail(TEMPO_HIP_E_ARG, "bad precision");
  LaunchCfg& lc = x->launch[precision == TEMPO_HIP_FP64 ? 1 : 0];
  switch (key) {
    case TEMPO_HIP_TUNE_SED_WAVE:
      if (value < 0 || value > 2) return fail(TEMPO_HIP_E_ARG, "sed_wave must be 0, 1 or 2");
      lc.sed_wave = value;
      return TEMPO_HIP_OK;
    case TEMPO_HIP_TUNE_BLOCK_A:
    case TEMPO_HIP_TUNE_BLOCK_C:
      if (value != 64 && value != 128 && value != 256) return fail(TEMPO_HIP_E_ARG, "block must be 64, 128 or 256");
      (key == TEMPO_HIP_TUNE_BLOCK_A ? lc.block_a : lc.block_c) = value;
      return TEMPO_HIP_OK;
    case TEMPO_HIP_TUNE_ORDER:
      if (value < -1 || value > 3) return fail(TEMPO_HIP_E_ARG, "order must be 0..3, or -1 (chosen)");
      lc.order = value;
      return TEMPO_HIP_OK;
    case TEMPO_HIP_TUNE_FUSED:
      if (value != 0 && value != 1) return fail(TEMPO_HIP_E_ARG, "fused must be 0 or 1");
      if (value == 1) return fail(TEMPO_HIP_E_UNSUPPORTED, "this library has no single-launch step");
      return TEMPO_HIP_OK;
    case TEMPO_HIP_TUNE_WAVES_A:
      if (value < -1 || value > 1) return fail(TEMPO_HIP_E_ARG, "waves_a must be 0 or 1, or -1 (chosen)");
      lc.waves_a = value;
      return TEMPO_HIP_OK;
    case TEMPO_HIP_TUNE_CCN_LDS:
      if (value != 0 && value != 1) return fail(TEMPO_HIP_E_ARG, "ccn_lds must be 0 or 1");
      lc.ccn_lds = value;
      return TEMPO_HIP_OK;
    case TEMPO_HIP_TUNE_HOST_SLABS:
      if (value < 0 || value > 4096) return fail(TEMPO_HIP_E_ARG, "host slabs must be 0..4096");
      lc.host_slabs = value;
      return TEMPO_HIP_OK;
    case TEMPO_HIP_TUNE_HOST_THREADS:
      if (value < 1 || value > 64) return fail(TEMPO_HIP_E_ARG, "host threads must be 1..64");
      lc.host_threads = value;
      return TEMPO_HIP_OK;
    default:
      return fail(TEMPO_HIP_E_ARG, "unknown tuning key");
  }
}

int tempo_hip_profile(tempo_hip_ctx* x, int enable) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  for (auto e : x->events) (void)hipEventDestroy(e);
  x->events.clear();
  x->profile = enable != 0;
  return TEMPO_HIP_OK;
}

int tempo_hip_profile_read(tempo_hip_ctx* x, double* ms, int n, int* runs) {
  if (!x || !ms || n < 4) return fail(TEMPO_HIP_E_ARG, "need room for 4 phases");
  for (int p = 0; p < 4; ++p) ms[p] = 0.0;
  const size_t nr = x->events.size() / 5;
  for (size_t r = 0; r < nr; ++r) {
    HIP_TRY(hipEventSynchronize(x->events[5 * r + 4]));
    for (int p = 0; p < 4; ++p) {
      float t = 0.f;
      HIP_TRY(hipEventElapsedTime(&t, x->events[5 * r + p], x->events[5 * r + p + 1]));
      ms[p] += t;
    }
  }
  if (runs) *runs = int(nr);
  return TEMPO_HIP_OK;
}

int tempo_hip_substeps(tempo_hip_ctx* x, int* out, size_t n) {
  if (!x || !out) return fail(TEMPO_HIP_E_ARG, "NULL argument");
  if (!x->last_ksub)
    return fail(TEMPO_HIP_E_ARG, "no substep record (no step yet, or the last step ran on host arrays in slabs)");
  if (n != size_t(10) * x->last_ncol && n != size_t(kSubRows) * x->last_ncol)
    return fail(TEMPO_HIP_E_ARG, "need 10*ncol or 12*ncol entries");
  HIP_TRY(hipMemcpy(out, x->last_ksub, n * sizeof(int), hipMemcpyDeviceToHost));
  return TEMPO_HIP_OK;
}

}  // extern "C"

namespace tempo {

int set_error(int code, const char* msg) { return fail(code, msg); }

// One step of tempo_hip_run with its per-point scratch carved from the
// caller's device block [base, base + bytes) of the context's device:
// nothing is allocated.  E_ARG when the batch needs more than bytes.
int run_with_scratch(tempo_hip_ctx* x, const tempo_hip_fields* f, const tempo_hip_diags* d, const tempo_hip_dims* dm,
                     double dt, int itimestep, int precision, void* stream, void* base, size_t bytes) {
  if (!x) return fail(TEMPO_HIP_E_ARG, "NULL context");
  int rc = check_run_args(f, dm, dt);
  if (rc) return ok_if_empty(rc);
  if (precision != TEMPO_HIP_FP32 && precision != TEMPO_HIP_FP64)
    return fail(TEMPO_HIP_E_ARG, "precision must be TEMPO_HIP_FP32 or TEMPO_HIP_FP64");
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev != x->device) return fail(TEMPO_HIP_E_ARG, "call with the context's device current");
  const bool r64 = precision == TEMPO_HIP_FP64;
  StepArgs<float> p32;
  StepArgs<double> p64;
  std::memset(&p32, 0, sizeof(p32));
  std::memset(&p64, 0, sizeof(p64));
  p32.ncol = p64.ncol = dm->ni * dm->nj;
  p32.nz = p64.nz = dm->nz;
  // the batches accepted are those of the stated bytes per point, which count
  // the wide copy above kSedLevels levels
  const ScratchSizes z = r64 ? step_scratch(x, p64, kSedLevels) : step_scratch(x, p32, kSedLevels);
  if (z.total() > bytes)
    return fail(TEMPO_HIP_E_ARG, std::to_string(p32.ncol) + " columns of " + std::to_string(p32.nz) +
                                     " levels need " + std::to_string(z.total()) + " bytes of scratch, more than the " +
                                     std::to_string(bytes) + " available");
  char* p = static_cast<char*>(base);
  auto take = [&](size_t b) -> void* {
    if (!b) return nullptr;
    void* q = p;
    p += ScratchSizes::up(b);
    return q;
  };
  ScratchPtrs sc;
  sc.sr = take(z.sr);
  sc.sd = take(z.sd);
  sc.pf = take(z.pf);
  sc.vt = take(z.vt);
  sc.cf = take(z.cf);
  sc.kmelt = take(z.kmelt);
  sc.precip = take(z.precip);
  sc.ksub = take(z.ksub);
  sc.semiw = take(z.semiw);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return r64 ? run_impl<double>(x, f, d, dm, dt, itimestep, s, nullptr, &sc)
             : run_impl<float>(x, f, d, dm, dt, itimestep, s, nullptr, &sc);
}

}  // namespace tempo
