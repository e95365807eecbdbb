// api.cpp -- libqcu.so C ABI: the five drop-in entry points of qcu.h and the
// extended API of qcu_ex.h, on top of the resident-field runtime.
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "qcu_host.h"
#include "qcu_shift_storage.h"

namespace qcu {

// ------------------------------------------------------------ errors ------
static int g_last_code = QCU_SUCCESS;
static std::string g_last_msg;

void check_hip(hipError_t e, const char* what, const char* file, int line) {
  if (e == hipSuccess) return;
  (void)hipGetLastError();  // reported here: left in place, it would fail the next call's launch check
  char buf[512];
  snprintf(buf, sizeof buf, "HIP error %d (%s) from %s at %s:%d", (int)e, hipGetErrorString(e), what, file, line);
  throw Error(e == hipErrorOutOfMemory ? QCU_ERROR_OUT_OF_MEMORY : QCU_ERROR_HIP, buf);
}

static void record(int code, const std::string& msg) {
  g_last_code = code;
  g_last_msg = msg;
}
void set_last_error(int code, const std::string& msg) { record(code, msg); }

template <typename F>
static int guarded(F&& f) {
  try {
    std::lock_guard<std::recursive_mutex> lk(ctx().mu);
    f();
    return QCU_SUCCESS;
  } catch (const Error& e) {
    record(e.code, e.what());
    return e.code;
  } catch (const std::bad_alloc&) {
    record(QCU_ERROR_OUT_OF_MEMORY, "host allocation failed");
    return QCU_ERROR_OUT_OF_MEMORY;
  } catch (const std::exception& e) {
    record(QCU_ERROR_STATE, e.what());
    return QCU_ERROR_STATE;
  }
}

// drop-in entry points report like the reference's checkCudaErrors: message on
// stderr, then exit(-1) unless QCU_EXIT_ON_ERROR=0
template <typename F>
static void dropin(const char* name, F&& f) {
  int rc = guarded(f);
  if (rc == QCU_SUCCESS) return;
  fprintf(stderr, "qcu: %s failed (error %d): %s\n", name, rc, g_last_msg.c_str());
  const char* env = getenv("QCU_EXIT_ON_ERROR");
  if (!(env && strcmp(env, "0") == 0)) exit(-1);
}

static bool quiet() {
  const char* e = getenv("QCU_QUIET");
  return e && strcmp(e, "0") != 0;
}

// ------------------------------------------------------------ buffers -----
DevBuf::~DevBuf() {
  if (p) (void)hipFree(p);
}
void DevBuf::release() {
  if (p) QHIP(hipFree(p));
  p = nullptr;
  n = 0;
}
// hipMalloc; when the card is full, what is only kept to save a later allocation (a changed
// drop-in gauge's old fields and solver workspace) is given back first
static void* device_malloc(size_t bytes) {
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e == hipErrorOutOfMemory) {
    bool freed = drop_unbound_batch();
    GaugeField* g = ctx().dropin.g.get();
    if (g && !g->spare.empty()) {
      g->spare.clear();
      freed = true;
    }
    if (freed) {
      (void)hipGetLastError();
      e = hipMalloc(&p, bytes);
    }
  }
  check_hip(e, "hipMalloc", __FILE__, __LINE__);
  return p;
}
void* DevBuf::alloc(size_t bytes) {
  release();
  if (bytes == 0) return nullptr;
  p = device_malloc(bytes);
  n = bytes;
  return p;
}
void DevBuf::ensure(size_t bytes) {
  if (bytes > n) alloc(bytes);
}

Context& ctx() {
  static Context c;
  return c;
}

DevBuf* Context::buf(const std::string& name, size_t bytes) {
  auto& slot = scratch[name];
  if (!slot) slot.reset(new DevBuf);
  if (slot->n < bytes) {
    QHIP(hipStreamSynchronize(stream));  // the old buffer may still be in use
    slot->alloc(bytes);
  }
  return slot.get();
}

void ensure_init() {
  Context& c = ctx();
  if (c.inited) return;
  int n = 0;
  QHIP(hipGetDeviceCount(&n));
  if (n <= 0) throw Error(QCU_ERROR_HIP, "no HIP device");
  QHIP(hipSetDevice(c.device));
  QHIP(hipStreamCreate(&c.stream));  // default priority, blocking w.r.t. the null stream
  noalloc_setup(c.device);           // device address of qcuHopNoAlloc's static scratch
  qcuDefaultSolveParams(&c.default_solve);
  c.default_solve.precision = QCU_PREC_DOUBLE;
  c.default_solve.tol = 1e-12;
  c.inited = true;
  load_tune_cache();
}

void validate_lattice(const int L[4]) {
  for (int i = 0; i < 4; ++i) QREQ(L[i] > 0, "lattice sizes must be positive");
  QREQ(L[0] % 2 == 0, "Lx must be even");
  double v = (double)L[0] * L[1] * L[2] * L[3];
  QREQ(v / 2 < 2147483647.0, "half volume must fit in 31 bits");
}

// --------------------------------------------------------- gauge fields ---
size_t GaugeField::bytes() const {
  size_t s = aos.n;
  for (auto& a : packed)
    for (auto& b : a) s += b.n;
  for (auto& kv : clovers)
    for (int p = 0; p < 3; ++p)
      for (int q = 0; q < 2; ++q) s += kv.second->A[p][q].n + kv.second->Ainv[p][q].n;
  for (auto& b : spare) s += b.n;
  return s;
}

void* GaugeField::take(DevBuf& b, size_t bytes) {
  for (auto it = spare.begin(); it != spare.end(); ++it)
    if (it->n == bytes) {
      b.swap(*it);
      spare.erase(it);
      return b.p;
    }
  return b.alloc(bytes);
}

void GaugeField::forget_links() {
  auto keep = [&](DevBuf& b) {
    if (!b.p) return;
    spare.emplace_back();
    spare.back().swap(b);
  };
  for (auto& a : packed)
    for (auto& b : a) keep(b);
  for (auto& kv : clovers)
    for (int p = 0; p < 3; ++p)
      for (int q = 0; q < 2; ++q) {
        keep(kv.second->A[p][q]);
        keep(kv.second->Ainv[p][q]);
      }
  clovers.clear();
}

// Fields are put together in buffers of their own and handed over once the launches that
// fill them are queued, so that a buffer a gauge or a clover field holds is always a built
// one: a step that throws (an allocation above all) leaves everything as it was.
const void* GaugeField::get(int prec, int recon) {
  DevBuf& b = packed[prec][recon == 12 ? 1 : 0];
  if (!b.p) {
    if (!aos.p && (prec == F64 || recon != 12)) throw Error(QCU_ERROR_STATE, "internal: drop-in links are recon-12");
    DevBuf d;
    take(d, gauge_bytes(prec, recon, geo.vh));
    if (aos.p) launch_gauge_pack(prec, recon, aos.p, d.p, geo.vh, stream());
    else launch_gauge_repack(prec, packed[F64][1].p, d.p, geo.vh, stream());
    QHIP(hipGetLastError());
    b.swap(d);
  }
  return b.p;
}

CloverField* GaugeField::clover(double ck, int prec, CloverParts parts) {
  std::unique_ptr<CloverField>& slot = clovers[ck];
  if (!slot) {
    slot.reset(new CloverField);
    slot->ck = ck;
    slot->vh = geo.vh;
  }
  CloverField* cf = slot.get();
  bool need_a[2], need_inv[2];
  for (int p = 0; p < 2; ++p) {
    const bool inv = parts == CLOVER_ALL || (parts == CLOVER_SOLVE && p == 1);
    need_a[p] = !cf->A[F64][p].p;
    need_inv[p] = inv && !cf->Ainv[F64][p].p;
  }
  const bool need[2] = {need_a[0] || need_inv[0], need_a[1] || need_inv[1]};
  if (need[0] || need[1]) {
    const size_t half = clover_bytes(F64, geo.vh) / 2;
    const int recon = aos.p ? 18 : 12;
    CloverBuild b;
    DevBuf A[2], Ainv[2], bad;
    b.gauge = get(F64, recon);
    for (int p = 0; p < 2; ++p) {
      b.A[p] = need_a[p] ? take(A[p], half) : nullptr;
      b.Ainv[p] = need_inv[p] ? take(Ainv[p], half) : nullptr;
    }
    const bool first_inv = (need_inv[0] || need_inv[1]) && !cf->bad.p;
    if (first_inv) {
      bad.alloc(sizeof(int));
      QHIP(hipMemsetAsync(bad.p, 0, sizeof(int), stream()));
    }
    b.nbad = static_cast<int*>(first_inv ? bad.p : cf->bad.p);
    b.ck = ck;
    b.only = need[0] && need[1] ? -1 : need[1];
    b.geo = geo;
    launch_clover_build(recon, b, stream());
    QHIP(hipGetLastError());
    for (int p = 0; p < 2; ++p) {
      if (need_a[p]) cf->A[F64][p].swap(A[p]);
      if (need_inv[p]) cf->Ainv[F64][p].swap(Ainv[p]);
    }
    if (first_inv) cf->bad.swap(bad);
  }
  // inner-precision parts: A_ee and A^-1_oo
  if (parts != CLOVER_A && prec != F64 && !cf->A[prec][0].p) {
    const size_t half = clover_bytes(prec, geo.vh) / 2;
    DevBuf A, Ainv;
    take(A, half);
    take(Ainv, half);
    launch_clover_convert(prec, cf->a(F64, 0), A.p, geo.vh, stream());
    launch_clover_convert(prec, cf->ainv(F64, 1), Ainv.p, geo.vh, stream());
    QHIP(hipGetLastError());
    cf->A[prec][0].swap(A);
    cf->Ainv[prec][1].swap(Ainv);
  }
  return cf;
}

static std::unique_ptr<GaugeField> new_gauge(const int L[4], bool keep_aos = true) {
  validate_lattice(L);
  std::unique_ptr<GaugeField> g(new GaugeField);
  for (int i = 0; i < 4; ++i) g->L[i] = L[i];
  g->geo = make_geom(L);
  if (keep_aos) g->aos.alloc((size_t)8 * g->geo.vh * 9 * 16);
  return g;
}

std::unique_ptr<GaugeField> make_gauge_from_aos(const void* aos_device, const int L[4]) {
  auto g = new_gauge(L);
  QHIP(hipMemcpyAsync(g->aos.p, aos_device, g->aos.n, hipMemcpyDeviceToDevice, stream()));
  return g;
}

std::unique_ptr<GaugeField> make_gauge_random(const int L[4], uint64_t seed, double eps) {
  auto g = new_gauge(L);
  launch_gauge_random(g->aos.p, g->geo.vh, seed, eps, stream());
  QHIP(hipGetLastError());
  return g;
}

// ------------------------------------------------------------- tuning -----
// "hop:prec:recon:vh:nrhs" for the plain epilogue, with ":e<epi>" for the others
std::string tune_key(int prec, int recon, long vh, int nrhs, int epi) {
  char b[96];
  if (epi == EPI_PLAIN) snprintf(b, sizeof b, "hop:%d:%d:%ld:%d", prec, recon, vh, nrhs);
  else snprintf(b, sizeof b, "hop:%d:%d:%ld:%d:e%d", prec, recon, vh, nrhs, epi);
  return b;
}
// the largest divisor of Lt up to an eighth of it (rounded up)
static int eighth_of_t(const Geom& geo) {
  int tt = (geo.L[3] + 7) / 8;
  while (geo.L[3] % tt) --tt;
  return tt;
}

// Whether a hop on internal fields takes the leg-split kernel (k_hop_split.inc) when no
// shape was tuned or pinned for it: while the launch's links and spinors come from the
// Infinity Cache, the split's four waves per chunk keep more of that latency in flight;
// past it the two kernels wait for the same HBM bytes, and the LDS kernel's one read of
// the links per batch wins.  Per launch, hop_kernel against this one (us): 8^4 FP64 9.2 /
// 5.1, FP32 6.9 / 4.2; 16^3x32 FP64 recon-18 20.2 / 17.3, FP32 10.9 / 7.4, FP16 9.4 / 6.4;
// 24^3x48 FP32 43.6 / 29.2 (190 MB), FP16 27 / 18.5; above the line 32^3x64 FP32 (600 MB)
// 113 / 127; FP64 recon-12 gains up to 509 MB (24^3x48 95 / 75) and is even at 1.2 GB.
// hop_lds_kernel against this one: 24^3x48 FP32 2 RHS (243 MB) 64 / 43, 3 RHS (303 MB) 74 /
// 90; 16^2x32x64 FP32 240 MB 66 / 46, recon-18 288 MB 70 / 82; 12^2x16x64 FP64 216 MB 59 /
// 52, 297 MB 83 / 107.  FP16 spends its time on unpacking and rebuilding the links, which
// the LDS kernel does once per batch: 24^3x48 4 RHS 61 / 62, 16^3x32 6 RHS 21 / 20, 12 RHS
// 33 / 36.
//
// A clover epilogue's clover is part of a single launch's data: clover solves of one source
// with hop_kernel / this (ms): FP32 24^3x48 (286 MB with the clover) 8.7 / 8.2, recon-18 (350)
// 9.9 / 10.5, 24^3x56 (334) 9.6 / 10.5, 28^3x48 (455) 12.9 / 13.4; FP64 recon-12 24^3x40 (477)
// 13.6 / 13.2, 24^3x48 (573) 15.7 / 15.8, 24^3x56 (668) 17.2 / 18.9, 24^3x64 (764) 19.5 / 20.7;
// without a clover FP32 28^3x48 (303) 10.1 / 9.9, 24^3x64 recon-18 (339) 9.9 / 10.1, FP64
// recon-12 26^3x56 (566) 18.0 / 17.8, 28^3x64 (809) 24.5 / 25.7.
// In a batch the clover is read once per right-hand side here, where the LDS kernel stages it
// once, and each after the second counts (solves, LDS kernel / this): FP64 16^3x32 4 RHS (237
// MB with the clover) 29.3 / 25.3, 6 (352) 36.6 / 39.1, 16^4 8 (239) 20.9 / 19.2, 16 (491) 37.1
// / 42.1, 20^3x40 2 (246) 48.1 / 38.8; FP32 20^3x40 3 (200) 28.0 / 27.3, 4 (276) 33.6 / 35.6,
// 16^3x32 6 (176) 20.9 / 18.5, 16 (491) 44.7 / 53.6.  FP16 counts none up to 3 RHS (24^3x48 50.9
// / 43.5, 24^3x64 19.1 / 17.8), and beyond them its line is 80 MB: 16^4 6 (46) 10.0 / 8.6, 12
// (94) 13.9 / 14.6, 16^3x32 8 (124) 18.1 / 18.7, 24^3x48 4 (297) 51.2 / 56.5.
static bool split_pays(int prec, int recon, long vh, int nrhs, int epi) {
  const bool clover = epi == EPI_CLOV || epi == EPI_CLOV_XPAY;
  const bool few16 = prec == F16 && nrhs <= 3;
  const int counted = !clover ? 0 : nrhs == 1 ? 1 : few16 ? 0 : nrhs - 2;
  const size_t bytes = gauge_bytes(prec, recon, vh) + 2 * (size_t)nrhs * spinor_bytes(prec, vh) +
                       (size_t)counted * (clover_bytes(prec, vh) / 2);
  if (bytes > ((size_t)(nrhs > 1 ? 256 : prec == F64 && recon == 12 ? 550 : 300) << 20)) return false;
  if (prec == F16 && clover) return few16 || bytes <= (size_t)80 << 20;
  return prec != F16 || nrhs <= 4 || (vh + 63) / 64 * nrhs <= 6144;
}
// t-slices its chunks are taken at a time (ChunkOrder): an eighth of Lt, one tile per XCD
// (16^3x32 FP64 4 RHS 40.4 -> 35.6 us, 24^3x48 FP32 33.4 -> 29.2), or storage order past
// the Infinity Cache (24^3x48 FP64 recon-12 75 us, 85 in tiles)
static int split_slices(const Geom& geo, size_t bytes) {
  if (bytes > ((size_t)256 << 20)) return 1;
  return eighth_of_t(geo);
}

// the shape tuned for this epilogue, else the one tuned for the plain epilogue, else
// the default
Tune tuned_hop(int prec, int recon, long vh, int nrhs, int epi) {
  auto it = ctx().tune.find(tune_key(prec, recon, vh, nrhs, epi));
  if (it != ctx().tune.end()) return it->second;
  it = ctx().tune.find(tune_key(prec, recon, vh, nrhs, EPI_PLAIN));
  if (it != ctx().tune.end()) return it->second;
  Tune t;
  t.split = split_pays(prec, recon, vh, nrhs, epi);
  if (nrhs > 1) {  // every right-hand side in one block per 64-site chunk, its links
    // staged in LDS once (hop_lds_kernel; on 32^3x64 with 12 right-hand sides 22-29 %
    // faster than the best shape sharing link loads within a wave), blocks round-robin over
    // the XCDs.  Four waves per block, of which FP32 and FP64 gain with two right-hand sides
    // already (32^3x64 2 RHS, two waves / four: FP32 184 / 175 us, FP64 421 / 376); FP16 two
    // while the links weigh more than the right-hand sides (2 RHS 104 / 128, 6 249 / 269, 12
    // 474 / 472, 24^3x48 6 RHS 80 / 85), or with a clover up to three of them (24^3x48 clover
    // solves of 4 RHS, two / four, 58.6 / 51.2 ms, 6 RHS 80.3 / 72.6).
    t.lds = 2;  // a clover shared by every right-hand side staged in LDS as well
    t.block = prec == F16 && nrhs <= (epi == EPI_CLOV || epi == EPI_CLOV_XPAY ? 3 : 6) ? 128 : 256;
    // and then eight waves where four leave a CU short of them: beside the clover an LDS
    // holds one block in FP64 and two in FP32.  32^3x64 four waves / eight: FP64 A^-1 D 5 RHS
    // 1,089 / 891 us, 12 1,762 / 1,687, its M^ 12 2,183 / 2,009; FP32 A^-1 D 12 RHS 856 / 815,
    // M^ 1,024 / 1,003, but with one right-hand side a wave 602 / 649 (8 RHS)
    t.clw = (prec == F64 && nrhs >= 5) || (prec == F32 && nrhs > 8) ? 8 : 0;
    t.xcd = 0;
    t.tz = -1;  // tiles of all of z by 8 t-planes, or launch_shape's chunk order where they
    t.tt = 8;   // do not fit
  }
  return t;
}
void set_tuned_hop(int prec, int recon, long vh, int nrhs, const Tune& t) {
  for (int e = EPI_PLAIN; e <= EPI_CLOV_XPAY; ++e) ctx().tune.erase(tune_key(prec, recon, vh, nrhs, e));
  ctx().tune[tune_key(prec, recon, vh, nrhs, EPI_PLAIN)] = t;
}

void launch_shape(int prec, int recon, int epi, HopArgs& a, const Tune& t, hipStream_t st) {
  if (t.split) {
    HopSplit s;
    s.h = a;
    s.drhs = FastDiv((uint32_t)a.nrhs);
    s.order = make_chunk_order(a.geo, split_slices(a.geo, gauge_bytes(prec, recon, a.geo.vh) +
                                                             2 * (size_t)a.nrhs * spinor_bytes(prec, a.geo.vh)));
    launch_hop_split(prec, recon, epi, s, st);
    return;
  }
  a.xcd_remap = t.xcd;
  a.gmajor = t.gm;
  a.rpw = t.rpw;
  a.spt = t.spt;
  a.cached = t.cached;
  a.lds = t.lds;
  a.walk = make_walk(a.geo, t.ty, t.tz < 0 ? a.geo.L[2] : t.tz, t.tt);
  a.order = make_chunk_order(a.geo, 1);
  a.clw = t.clw;
  // planes that are no whole chunks: t-slices in eighths of Lt, one per XCD, instead of
  // storage order round-robin.  24^3x48 12 RHS FP32 327 -> 270 us, FP64 708 -> 560, FP16 166
  // -> 147, 20^2x24x40 FP32 193 -> 151, FP64 399 -> 324, 24x20x32x48 3 RHS FP32 93 -> 77
  if (t.lds && (t.tz < 0 || t.order) && !a.walk.tile_z) {
    a.order = make_chunk_order(a.geo, eighth_of_t(a.geo));
    a.xcd_remap = 1;
  }
  launch_hop(prec, recon, epi, a, t.block, t.rb, t.rpt, st);
}

void hop(GaugeField& g, int prec, int recon, int epi, int parity, int dagger, double tbc, Vec in, Vec out, Vec x,
         const void* clov, double coef, int nrhs, double* partials, hipStream_t st) {
  QREQ(nrhs >= 1 && nrhs <= kMaxRhs, "nrhs out of range");
  const void* cl[kMaxRhs];
  double co[kMaxRhs];
  for (int r = 0; r < nrhs; ++r) {
    cl[r] = clov;
    co[r] = coef;
  }
  hop_v(g, prec, recon, epi, parity, dagger, tbc, in, out, x, cl, co, nrhs, partials, st);
}

void hop_v(GaugeField& g, int prec, int recon, int epi, int parity, int dagger, double tbc, Vec in, Vec out, Vec x,
           const void* const* clovs, const double* coefs, int nrhs, double* partials, hipStream_t st) {
  QREQ(nrhs >= 1 && nrhs <= kMaxRhs, "nrhs out of range");
  HopArgs a;
  memset(&a, 0, sizeof a);
  a.in = in.p;
  a.out = out.p;
  a.x = x.p;
  a.in_stride = in.stride;
  a.out_stride = out.stride;
  a.x_stride = x.stride;
  a.gauge = g.get(prec, recon);
  a.clov_shared = 1;
  for (int r = 0; r < nrhs; ++r) {
    a.clov[r] = clovs[r];
    a.coef[r] = coefs[r];
    if (clovs[r] != clovs[0]) a.clov_shared = 0;
  }
  a.partials = partials;
  a.geo = g.geo;
  a.parity = parity;
  a.dagger = dagger;
  a.tbc = tbc;
  a.nrhs = nrhs;
  const Tune t = tuned_hop(prec, recon, g.geo.vh, nrhs, epi);
  launch_shape(prec, recon, epi, a, t, st);
}

// t-slices the chunks of an interface launch are taken at a time (ChunkOrder): an eighth
// of Lt, so that each XCD's range is whole tiles and a chunk's t neighbours run beside
// it -- the largest divisor of Lt up to that.  One FP64 half spinor stays in storage
// order.  Storage order against this one, whole calls: 24^3x48 12-RHS FP32 732 / 618 us,
// FP32 62.9 / 55.1, FP16 57.2 / 48.9, full clover operator 234 / 226; 32^3x64 full clover
// operator 812 / 675; but one FP64 half spinor 84.7 / 91.7 and 264.6 / 269.6 us.
static int iface_slices(const Geom& geo, const IfaceHop& p, int nrhs) {
  if (p.prec == F64 && nrhs == 1 && p.parity >= 0) return 1;
  return eighth_of_t(geo);
}

bool hop_iface(const Geom& geo, const IfaceHop& p, int nrhs, void* const* out, const void* const* in, hipStream_t st) {
  QREQ(nrhs >= 1 && nrhs <= kMaxRhs, "nrhs out of range");
  const size_t n = (size_t)geo.vh * 192 * (p.parity < 0 ? 2 : 1);
  for (int r = 0; r < nrhs; ++r)
    for (int k = 0; k < nrhs; ++k) {
      const char* o = static_cast<const char*>(out[r]);
      const char* i = static_cast<const char*>(in[k]);
      const char* o2 = static_cast<const char*>(out[k]);
      if (o < i + n && i < o + n) return false;
      if (k != r && o < o2 + n && o2 < o + n) return false;
    }
  IfaceArgs a;
  a.gauge = p.links;
  a.clov0 = p.clov[0];
  a.clov1 = p.clov[1];
  a.tbc = p.tbc;
  a.coef = p.coef;
  a.parity = p.parity;
  a.drhs = FastDiv((uint32_t)nrhs);
  a.order = make_chunk_order(geo, iface_slices(geo, p, nrhs));
  a.geo = geo;
  for (int r = 0; r < nrhs; ++r) {
    a.in[r] = in[r];
    a.out[r] = out[r];
  }
  launch_hop_iface(p.prec, p.recon, p.epi, p.dagger, a, st);
  QHIP(hipGetLastError());
  return true;
}

}  // namespace qcu

using namespace qcu;

// =================================================================== qcu.h ===
static QcuParam g_param;

// 1: the drop-in calls trust that a gauge pointer they have seen still holds the same
// links (the copy is remade only by initGridSize / loadQcuGauge or a new pointer)
static bool dropin_trust_pointer() {
  const char* e = getenv("QCU_DROPIN_GAUGE_CACHE");
  return e && strcmp(e, "0") != 0;
}

static void require_aligned(const void* p, const char* what) {
  QREQ((reinterpret_cast<uintptr_t>(p) & 15) == 0, std::string(what) + " must be 16-byte aligned (complex128)");
}

static bool overlap(const void* a, const void* b, size_t n) {
  const char* x = static_cast<const char*>(a);
  const char* y = static_cast<const char*>(b);
  return x < y + n && y < x + n;
}

static uint64_t* fingerprint_parts() {
  uint64_t*& h = ctx().dropin.fp_parts;
  if (!h)
    QHIP(hipHostMalloc(reinterpret_cast<void**>(&h), kFingerprintBlocks * sizeof(uint64_t), hipHostMallocDefault));
  return h;
}
// the fingerprint last queued, once the library stream has been synchronised
static uint64_t fingerprint_value() {
  uint64_t h = 0;
  for (int k = 0; k < kFingerprintBlocks; ++k) h += ctx().dropin.fp_parts[k];
  return h;
}
// after a synchronisation of the library stream: take over the fingerprint of an import
static void dropin_settle() {
  Context::Dropin& d = ctx().dropin;
  if (d.fp_queued) d.fp = fingerprint_value();
  d.fp_queued = false;
}

// remake the drop-in copy from the caller's gauge: rows 0-1 packed, with their fingerprint,
// in one pass (16^3x32: 25 us; the copy, the rebuilt row, two packed forms and the
// fingerprint it replaces took 170)
static void dropin_rebuild(void* gauge, const QcuParam* param, bool same_geom) {
  Context::Dropin& d = ctx().dropin;
  if (d.g) QHIP(hipStreamSynchronize(stream()));
  d.ptr = nullptr;  // until the new links are in
  if (same_geom) {  // new links, no packed copies, no clover, in the old allocations
    unbind_cached_batches(d.g.get());
    d.g->forget_links();
  } else {
    if (d.g) drop_cached_batches(d.g.get());
    d.g.reset();
    d.g = new_gauge(param->lattice_size, false);
  }
  GaugeField& g = *d.g;
  g.take(g.packed[F64][1], gauge_bytes(F64, 12, g.geo.vh));
  launch_gauge_import(gauge, g.packed[F64][1].p, fingerprint_parts(), g.geo.vh, stream());
  QHIP(hipGetLastError());
  d.fp_queued = true;
  d.ptr = gauge;
}

// The packed copy and clover fields behind fullDslashQcu and cg_inverter.  The
// reference reads the caller's gauge on every call (src/dslash.cu:73,
// src/cg_inverter.cu:312-339), so a caller may change links in place between calls
// (an HMC update, smearing) or pass a reused address.  The copy is therefore checked
// against a fingerprint of the caller's buffer on every call -- one read of the gauge
// -- and remade, with its clover fields and solver state dropped, when it differs.
// QCU_DROPIN_GAUGE_CACHE=1 skips the check.  One copy is kept: a new pointer or
// geometry replaces it.  With `deferred` (fullDslashQcu), a copy that exists for this
// pointer and geometry is returned at once and the fingerprint is only queued: the
// caller runs its work, synchronises, and asks dropin_gauge_changed whether to redo it
// with a remade copy, which saves a synchronisation in the common case.
static GaugeField& dropin_gauge(void* gauge, const QcuParam* param, bool reload, bool* deferred = nullptr) {
  Context& c = ctx();
  if (deferred) *deferred = false;
  QREQ(gauge != nullptr, "gauge pointer is NULL");
  QREQ(param != nullptr, "QcuParam pointer is NULL");
  require_aligned(gauge, "gauge");
  validate_lattice(param->lattice_size);
  Context::Dropin& d = c.dropin;
  const bool same_geom = d.g && memcmp(d.g->L, param->lattice_size, sizeof(int) * 4) == 0;
  const bool same = same_geom && d.ptr == gauge;
  if (same && !reload && dropin_trust_pointer()) return *d.g;
  if (d.fp_queued) {  // an import whose caller did not get to settle it
    QHIP(hipStreamSynchronize(stream()));
    dropin_settle();
  }
  if (same && !reload) {
    launch_fingerprint(gauge, fingerprint_parts(), d.g->geo.vh, stream());
    QHIP(hipGetLastError());
    if (deferred) {
      *deferred = true;
      return *d.g;
    }
    QHIP(hipStreamSynchronize(stream()));
    if (fingerprint_value() == d.fp) return *d.g;
  }
  dropin_rebuild(gauge, param, same_geom);
  return *d.g;
}

// after a deferred dropin_gauge and a synchronisation of the library stream: true
// when the caller's gauge had changed, in which case the copy has been remade and the
// caller redoes its work
static bool dropin_gauge_changed(void* gauge, const QcuParam* param) {
  if (fingerprint_value() == ctx().dropin.fp) return false;
  dropin_rebuild(gauge, param, true);
  return true;
}

extern "C" void initGridSize(QcuGrid_t* grid, QcuParam* p_param, void* gauge, void* fermion_in, void* fermion_out) {
  (void)fermion_in;
  (void)fermion_out;
  dropin("initGridSize", [&] {
    ensure_init();
    QREQ(grid && p_param, "initGridSize: NULL argument");
    for (int i = 0; i < 4; ++i)
      QREQ(grid->grid_size[i] == 1, "initGridSize: this build keeps the lattice on one GPU (grid_size must be 1,1,1,1)");
    validate_lattice(p_param->lattice_size);
    Context& c = ctx();
    memcpy(c.L, p_param->lattice_size, sizeof c.L);
    c.have_geom = true;
    g_param = *p_param;
    if (gauge) {
      dropin_gauge(gauge, p_param, true);
      QHIP(hipStreamSynchronize(stream()));
      dropin_settle();
    }
  });
}

extern "C" void loadQcuGauge(void* gauge, QcuParam* param) {
  dropin("loadQcuGauge", [&] {
    ensure_init();
    dropin_gauge(gauge, param, true);
    QHIP(hipStreamSynchronize(stream()));
    dropin_settle();
  });
}

// One kernel on the caller's buffers: the gauge is read on every call, as the
// reference's returned value (mpiDslashNaive) reads it, so no copy or fingerprint is
// needed here.
extern "C" void dslashQcu(void* fermion_out, void* fermion_in, void* gauge, QcuParam* param, int parity) {
  dropin("dslashQcu", [&] {
    ensure_init();
    QREQ(parity == 0 || parity == 1, "dslashQcu: parity must be 0 or 1");
    QREQ(fermion_out && fermion_in && gauge && param, "dslashQcu: NULL argument");
    require_aligned(fermion_in, "fermion_in");
    require_aligned(fermion_out, "fermion_out");
    require_aligned(gauge, "gauge");
    validate_lattice(param->lattice_size);
    const Geom g = make_geom(param->lattice_size);
    const char* i = static_cast<const char*>(fermion_in);
    char* o = static_cast<char*>(fermion_out);
    QREQ(o + g.vh * 192 <= i || i + g.vh * 192 <= o, "dslashQcu: fermion_out and fermion_in overlap");
    launch_dslash(fermion_in, fermion_out, gauge, g, parity, stream());
    QHIP(hipGetLastError());
    QHIP(hipStreamSynchronize(stream()));
  });
}

extern "C" void fullDslashQcu(void* fermion_out, void* fermion_in, void* gauge, QcuParam* param, int dagger_flag) {
  dropin("fullDslashQcu", [&] {
    ensure_init();
    QREQ(fermion_out && fermion_in, "fullDslashQcu: NULL spinor");
    require_aligned(fermion_in, "fermion_in");
    require_aligned(fermion_out, "fermion_out");
    bool deferred = false;
    GaugeField& g = dropin_gauge(gauge, param, false, &deferred);
    if (deferred && overlap(fermion_out, fermion_in, (size_t)2 * g.geo.vh * 192)) {
      // what overwrites its input cannot be redone: the fingerprint is looked at first
      QHIP(hipStreamSynchronize(stream()));
      dropin_gauge_changed(gauge, param);
      deferred = false;
    }
    qcuOperator op = {1.0, 1.0, 1, 12};
    apply_m_iface(g, op, fermion_out, fermion_in, dagger_flag ? 1 : 0);
    QHIP(hipStreamSynchronize(stream()));
    if (deferred && dropin_gauge_changed(gauge, param)) {  // the links changed in place: redo
      apply_m_iface(*ctx().dropin.g, op, fermion_out, fermion_in, dagger_flag ? 1 : 0);
      QHIP(hipStreamSynchronize(stream()));
    }
    dropin_settle();
  });
}

extern "C" void cg_inverter(void* b_vector, void* x_vector, void* gauge, QcuParam* param) {
  qcuSolveStats st;
  memset(&st, 0, sizeof st);
  // A solve that stops at max_iter (or breaks down) is not an error of the call: like
  // the reference (src/cg_inverter.cu:331-345) it leaves the last iterate in x and
  // prints cg_failed!!!; qcuGetLastError() then returns QCU_ERROR_NOT_CONVERGED (or
  // QCU_ERROR_BREAKDOWN).  The solve has synchronised by then.
  int rc = guarded([&] {
    ensure_init();
    QREQ(b_vector && x_vector, "cg_inverter: NULL spinor");
    require_aligned(b_vector, "b_vector");
    require_aligned(x_vector, "x_vector");
    GaugeField& g = dropin_gauge(gauge, param, false);
    qcuOperator op = {1.0, 1.0, 1, 12};
    void* xs[1] = {x_vector};
    const void* bs[1] = {b_vector};
    solve_batch(g, op, ctx().default_solve, 1, xs, bs, &st);
    QHIP(hipStreamSynchronize(stream()));
    dropin_settle();
  });
  if (rc != QCU_SUCCESS && rc != QCU_ERROR_NOT_CONVERGED && rc != QCU_ERROR_BREAKDOWN) {
    const std::string msg = g_last_msg;
    dropin("cg_inverter", [&] { throw Error(rc, msg); });
  }
  if (!quiet()) {
    // the reference's progress lines (src/cg_inverter.cu:330,342-349)
    if (st.converged) printf("number of iteration %d\ncg success!!!\n", st.iterations);
    else printf("cg_failed!!!\n");
    printf("true residual ||b - M x|| / ||b|| = %.3e\n", st.true_residual);
  }
}

// ==================================================== qcu_shift_storage.h ===
// [a, a + na) and [b, b + nb) must not overlap
static void require_disjoint(const void* a, size_t na, const void* b, size_t nb, const char* who) {
  const char* x = static_cast<const char*>(a);
  const char* y = static_cast<const char*>(b);
  QREQ(x + na <= y || y + nb <= x, std::string(who) + ": dst and src overlap");
}

// kind 0: one half spinor, kind 1: a gauge (src/qcu_shift_storage.cu:166-194)
static void shift_storage(const char* who, int kind, void* dst, void* src, int dir, int Lx, int Ly, int Lz, int Lt) {
  ensure_init();
  QREQ(dst && src, std::string(who) + ": NULL pointer");
  QREQ(dir == TO_COALESCE || dir == TO_NON_COALESCE, std::string(who) + ": shift_direction must be 0 or 1");
  const int L[4] = {Lx, Ly, Lz, Lt};
  validate_lattice(L);
  long vh = (long)Lx * Ly * Lz * Lt / 2;
  size_t aos = (size_t)vh * (kind == 0 ? 24 : 8 * 18) * 8;
  size_t soa = (size_t)vh * (kind == 0 ? 24 : 8 * 12) * 8;
  const bool to_soa = dir == TO_COALESCE;
  require_disjoint(dst, to_soa ? soa : aos, src, to_soa ? aos : soa, who);
  launch_shift_storage(kind, to_soa, src, dst, vh, stream());
  QHIP(hipGetLastError());
  QHIP(hipStreamSynchronize(stream()));
}

extern "C" void shiftVectorStorage(void* dst_vec, void* src_vec, int shift_direction, int Lx, int Ly, int Lz, int Lt) {
  dropin("shiftVectorStorage",
         [&] { shift_storage("shiftVectorStorage", 0, dst_vec, src_vec, shift_direction, Lx, Ly, Lz, Lt); });
}

extern "C" void shiftGaugeStorage(void* dst_vec, void* src_vec, int shift_direction, int Lx, int Ly, int Lz, int Lt) {
  dropin("shiftGaugeStorage",
         [&] { shift_storage("shiftGaugeStorage", 1, dst_vec, src_vec, shift_direction, Lx, Ly, Lz, Lt); });
}

// ================================================================ qcu_ex.h ===
extern "C" {

static int lex_eo(const char* who, int to_eo, void* dst, const void* src, const int L[4], int field) {
  return guarded([&] {
    ensure_init();
    QREQ(dst && src && L, std::string(who) + ": NULL argument");
    QREQ(field == QCU_FIELD_SPINOR || field == QCU_FIELD_GAUGE, std::string(who) + ": field must be spinor or gauge");
    validate_lattice(L);
    long vol = (long)L[0] * L[1] * L[2] * L[3];
    QREQ(vol < 2147483648L, std::string(who) + ": volume must be below 2^31 sites");
    int nc = field == QCU_FIELD_SPINOR ? 12 : 9, nf = field == QCU_FIELD_SPINOR ? 1 : 4;
    const size_t n = (size_t)vol * nc * nf * 16;
    require_disjoint(dst, n, src, n, who);
    launch_lex_eo(to_eo, src, dst, L, nc, nf, stream());
    QHIP(hipGetLastError());
    QHIP(hipStreamSynchronize(stream()));
  });
}

int qcuLexToEvenOdd(void* eo, const void* lex, const int L[4], int field) {
  return lex_eo("qcuLexToEvenOdd", 1, eo, lex, L, field);
}
int qcuEvenOddToLex(void* lex, const void* eo, const int L[4], int field) {
  return lex_eo("qcuEvenOddToLex", 0, lex, eo, L, field);
}

int qcuInit(int device) {
  return guarded([&] {
    Context& c = ctx();
    if (c.inited && c.device != device) throw Error(QCU_ERROR_STATE, "qcuInit: already initialised on another device");
    c.device = device;
    ensure_init();
  });
}

int qcuFinalize(void) {
  return guarded([&] {
    Context& c = ctx();
    if (!c.inited) return;
    QHIP(hipStreamSynchronize(c.stream));
    drop_cached_batches(nullptr);
    c.dropin.g.reset();
    c.dropin.ptr = nullptr;
    c.dropin.fp_queued = false;
    c.scratch.clear();
    QHIP(hipStreamDestroy(c.stream));
    c.stream = nullptr;
    c.inited = false;
  });
}

int qcuGetLastError(void) { return g_last_code; }
const char* qcuGetLastErrorString(void) { return g_last_msg.c_str(); }
void qcuClearLastError(void) { record(QCU_SUCCESS, ""); }
const char* qcuVersion(void) { return "qcu-mi355x 0.1 (gfx950)"; }

int qcuMalloc(void** ptr, size_t bytes) {
  return guarded([&] {
    ensure_init();
    QREQ(ptr, "qcuMalloc: NULL");
    *ptr = nullptr;
    *ptr = device_malloc(bytes);
  });
}
int qcuFree(void* ptr) {
  return guarded([&] {
    ensure_init();
    QHIP(hipStreamSynchronize(stream()));
    QHIP(hipFree(ptr));
  });
}
int qcuMemcpyHtoD(void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    ensure_init();
    QHIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream()));
    QHIP(hipStreamSynchronize(stream()));
  });
}
int qcuMemcpyDtoH(void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    ensure_init();
    QHIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream()));
    QHIP(hipStreamSynchronize(stream()));
  });
}
int qcuMemcpyDtoD(void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    ensure_init();
    QHIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, stream()));
    QHIP(hipStreamSynchronize(stream()));
  });
}
int qcuMemset(void* dst, int value, size_t bytes) {
  return guarded([&] {
    ensure_init();
    QHIP(hipMemsetAsync(dst, value, bytes, stream()));
    QHIP(hipStreamSynchronize(stream()));
  });
}
int qcuSynchronize(void) {
  return guarded([&] {
    ensure_init();
    QHIP(hipStreamSynchronize(stream()));
  });
}
int qcuMemInfo(size_t* free_bytes, size_t* total_bytes) {
  return guarded([&] {
    ensure_init();
    QHIP(hipMemGetInfo(free_bytes, total_bytes));
  });
}

int qcuGaugeCreate(qcuGauge* out, const void* gauge, const int lattice_size[4]) {
  return guarded([&] {
    ensure_init();
    QREQ(out && gauge && lattice_size, "qcuGaugeCreate: NULL argument");
    auto g = make_gauge_from_aos(gauge, lattice_size);
    QHIP(hipStreamSynchronize(stream()));
    *out = reinterpret_cast<qcuGauge>(g.release());
  });
}
int qcuGaugeCreateRandom(qcuGauge* out, const int lattice_size[4], uint64_t seed, double eps) {
  return guarded([&] {
    ensure_init();
    QREQ(out && lattice_size, "qcuGaugeCreateRandom: NULL argument");
    QREQ(eps >= 0.0, "eps must be >= 0");
    auto g = make_gauge_random(lattice_size, seed, eps);
    QHIP(hipStreamSynchronize(stream()));
    *out = reinterpret_cast<qcuGauge>(g.release());
  });
}
int qcuGaugeDestroy(qcuGauge h) {
  return guarded([&] {
    ensure_init();
    QHIP(hipStreamSynchronize(stream()));
    drop_cached_batches(reinterpret_cast<GaugeField*>(h));
    delete reinterpret_cast<GaugeField*>(h);
  });
}
int qcuGaugeExport(qcuGauge h, void* gauge) {
  return guarded([&] {
    ensure_init();
    QREQ(h && gauge, "qcuGaugeExport: NULL argument");
    GaugeField& g = *reinterpret_cast<GaugeField*>(h);
    QHIP(hipMemcpyAsync(gauge, g.aos.p, g.aos.n, hipMemcpyDeviceToDevice, stream()));
    QHIP(hipStreamSynchronize(stream()));
  });
}
int qcuCloverExport(qcuGauge h, const qcuOperator* op, void* A, void* Ainv, int* nfallback) {
  return guarded([&] {
    ensure_init();
    QREQ(h && op, "qcuCloverExport: NULL argument");
    GaugeField& g = *reinterpret_cast<GaugeField*>(h);
    CloverField* cf = g.clover(op->kappa * op->csw, F64, CLOVER_ALL);
    size_t half = (size_t)g.geo.vh * 72 * 16;
    for (int p = 0; p < 2; ++p) {
      if (A) launch_clover_unpack(cf->a(F64, p), static_cast<char*>(A) + p * half, g.geo.vh, stream());
      if (Ainv) launch_clover_unpack(cf->ainv(F64, p), static_cast<char*>(Ainv) + p * half, g.geo.vh, stream());
    }
    QHIP(hipGetLastError());
    int nbad = 0;
    QHIP(hipMemcpyAsync(&nbad, cf->bad.p, sizeof(int), hipMemcpyDeviceToHost, stream()));
    QHIP(hipStreamSynchronize(stream()));
    if (nfallback) *nfallback = nbad;
  });
}

int qcuSourceGaussian(void* v, const int L[4], uint64_t seed) {
  return guarded([&] {
    ensure_init();
    QREQ(v && L, "qcuSourceGaussian: NULL argument");
    validate_lattice(L);
    long n = (long)L[0] * L[1] * L[2] * L[3] * 12;
    launch_source_gauss(v, n, seed, stream());
    QHIP(hipGetLastError());
    QHIP(hipStreamSynchronize(stream()));
  });
}

int qcuSourcePoint(void* v, const int L[4], const int coords[4], int spin, int colour) {
  return guarded([&] {
    ensure_init();
    QREQ(v && L && coords, "qcuSourcePoint: NULL argument");
    validate_lattice(L);
    QREQ(spin >= 0 && spin < 4 && colour >= 0 && colour < 3, "spin must be 0..3 and colour 0..2");
    for (int i = 0; i < 4; ++i) QREQ(coords[i] >= 0 && coords[i] < L[i], "coordinate outside the lattice");
    long vh = (long)L[0] * L[1] * L[2] * L[3] / 2;
    int parity = (coords[0] + coords[1] + coords[2] + coords[3]) & 1;
    long idx = (((long)coords[3] * L[2] + coords[2]) * L[1] + coords[1]) * (L[0] / 2) + coords[0] / 2;
    long off = ((parity * vh + idx) * 12 + spin * 3 + colour) * 16;
    static const double one[2] = {1.0, 0.0};
    QHIP(hipMemsetAsync(v, 0, (size_t)2 * vh * 192, stream()));
    QHIP(hipMemcpyAsync(static_cast<char*>(v) + off, one, 16, hipMemcpyHostToDevice, stream()));
    QHIP(hipStreamSynchronize(stream()));
  });
}

int qcuHop(qcuGauge h, void* out, const void* in, int parity, int dagger, int t_boundary, int recon, int precision) {
  return guarded([&] {
    ensure_init();
    QREQ(h && out && in, "qcuHop: NULL argument");
    QREQ(parity == 0 || parity == 1, "parity must be 0 or 1");
    QREQ(recon == 12 || recon == 18, "recon must be 12 or 18");
    QREQ(precision >= 0 && precision <= 2, "bad precision");
    QREQ(t_boundary == 1 || t_boundary == -1, "t_boundary must be +1 or -1");
    GaugeField& g = *reinterpret_cast<GaugeField*>(h);
    long vh = g.geo.vh;
    const IfaceHop p = {g.get(precision, recon), precision, recon, EPI_PLAIN, parity, dagger ? 1 : 0,
                        (double)t_boundary, 1.0, {nullptr, nullptr}};
    if (!hop_iface(g.geo, p, 1, &out, &in, stream())) {  // in and out overlap: staged
      DevBuf* a = ctx().buf("hop_in", spinor_bytes(F64, vh));
      DevBuf* b = ctx().buf("hop_out", spinor_bytes(F64, vh));
      launch_spinor_from_aos(precision, in, 0, vec(a->p), vh, 1, stream());
      hop(g, precision, recon, EPI_PLAIN, parity, dagger ? 1 : 0, (double)t_boundary, vec(a->p), vec(b->p),
          vec(nullptr), nullptr, 1.0, 1, nullptr, stream());
      launch_spinor_to_aos(precision, vec(b->p), out, 0, vh, 1, stream());
    }
    QHIP(hipGetLastError());
    QHIP(hipStreamSynchronize(stream()));
  });
}

int qcuHopBatch(qcuGauge h, int nrhs, void* const* out, const void* const* in, int parity, int dagger,
                int t_boundary, int recon, int precision) {
  return guarded([&] {
    ensure_init();
    QREQ(h && out && in, "qcuHopBatch: NULL argument");
    QREQ(nrhs >= 1 && nrhs <= kMaxRhs, "nrhs out of range (1..16)");
    QREQ(parity == 0 || parity == 1, "parity must be 0 or 1");
    QREQ(recon == 12 || recon == 18, "recon must be 12 or 18");
    QREQ(precision >= 0 && precision <= 2, "bad precision");
    QREQ(t_boundary == 1 || t_boundary == -1, "t_boundary must be +1 or -1");
    for (int r = 0; r < nrhs; ++r) QREQ(out[r] && in[r], "qcuHopBatch: NULL spinor");
    GaugeField& g = *reinterpret_cast<GaugeField*>(h);
    long vh = g.geo.vh;
    const IfaceHop p = {g.get(precision, recon), precision, recon, EPI_PLAIN, parity, dagger ? 1 : 0,
                        (double)t_boundary, 1.0, {nullptr, nullptr}};
    if (!hop_iface(g.geo, p, nrhs, out, in, stream())) {  // an output overlaps an input: staged
      long fb = (long)spinor_bytes(precision, vh);
      DevBuf* a = ctx().buf("hopb_in", (size_t)fb * nrhs);
      DevBuf* b = ctx().buf("hopb_out", (size_t)fb * nrhs);
      for (int r = 0; r < nrhs; ++r) launch_spinor_from_aos(precision, in[r], 0, vec(a->c() + r * fb), vh, 1, stream());
      hop(g, precision, recon, EPI_PLAIN, parity, dagger ? 1 : 0, (double)t_boundary, vec(a->p, fb), vec(b->p, fb),
          vec(nullptr), nullptr, 1.0, nrhs, nullptr, stream());
      for (int r = 0; r < nrhs; ++r) launch_spinor_to_aos(precision, vec(b->c() + r * fb), out[r], 0, vh, 1, stream());
    }
    QHIP(hipGetLastError());
    QHIP(hipStreamSynchronize(stream()));
  });
}

int qcuApplyM(qcuGauge h, const qcuOperator* op, void* out, const void* in, int dagger) {
  return guarded([&] {
    ensure_init();
    QREQ(h && op && out && in, "qcuApplyM: NULL argument");
    apply_m_iface(*reinterpret_cast<GaugeField*>(h), *op, out, in, dagger ? 1 : 0);
    QHIP(hipStreamSynchronize(stream()));
  });
}

int qcuApplyComposite(qcuGauge h, const qcuOperator* op, int kind, void* out, const void* in, int dagger) {
  return guarded([&] {
    ensure_init();
    QREQ(h && op && out && in, "qcuApplyComposite: NULL argument");
    apply_composite_iface(*reinterpret_cast<GaugeField*>(h), *op, kind, out, in, dagger ? 1 : 0);
    QHIP(hipStreamSynchronize(stream()));
  });
}

int qcuApplyMhat(qcuGauge h, const qcuOperator* op, void* out, const void* in, int dagger, int precision) {
  return guarded([&] {
    ensure_init();
    QREQ(h && op && out && in, "qcuApplyMhat: NULL argument");
    QREQ(precision >= 0 && precision <= 2, "bad precision");
    apply_mhat_iface(*reinterpret_cast<GaugeField*>(h), *op, out, in, dagger ? 1 : 0, precision);
    QHIP(hipStreamSynchronize(stream()));
  });
}

void qcuDefaultSolveParams(qcuSolveParams* sp) {
  if (!sp) return;
  sp->tol = 1e-10;
  sp->max_iter = 0;
  sp->precision = QCU_PREC_SINGLE;
  sp->delta = 0.0;  // by inner precision: 1e-3 for FP32, 0.1 for FP16
  sp->graph = 1;
  sp->chunk = 8;
}

int qcuSetDefaultSolve(const qcuSolveParams* sp) {
  return guarded([&] {
    ensure_init();
    QREQ(sp, "qcuSetDefaultSolve: NULL");
    ctx().default_solve = *sp;
  });
}

int qcuSolve(qcuGauge h, const qcuOperator* op, const qcuSolveParams* sp, void* x, const void* b,
             qcuSolveStats* stats) {
  return guarded([&] {
    ensure_init();
    QREQ(h && op && sp && x && b, "qcuSolve: NULL argument");
    void* xs[1] = {x};
    const void* bs[1] = {b};
    solve_batch(*reinterpret_cast<GaugeField*>(h), *op, *sp, 1, xs, bs, stats);
  });
}

int qcuSolveBatch(qcuGauge h, const qcuOperator* op, const qcuSolveParams* sp, int nrhs, void* const* x,
                  const void* const* b, qcuSolveStats* stats) {
  return guarded([&] {
    ensure_init();
    QREQ(h && op && sp && x && b, "qcuSolveBatch: NULL argument");
    QREQ(nrhs >= 1 && nrhs <= kMaxRhs, "nrhs out of range (1..16)");
    solve_batch(*reinterpret_cast<GaugeField*>(h), *op, *sp, nrhs, x, b, stats);
  });
}

int qcuBenchHop(qcuGauge h, int precision, int recon, int nrhs, int iters, double* ms) {
  return guarded([&] {
    ensure_init();
    QREQ(h && ms && iters > 0, "qcuBenchHop: bad argument");
    QREQ(nrhs >= 1 && nrhs <= kMaxRhs, "nrhs out of range");
    GaugeField& g = *reinterpret_cast<GaugeField*>(h);
    long vh = g.geo.vh;
    size_t fb = spinor_bytes(precision, vh);
    DevBuf* src = ctx().buf("bench_src", (size_t)vh * 192 * nrhs);
    DevBuf* a = ctx().buf("bench_a", fb * nrhs);
    DevBuf* b = ctx().buf("bench_b", fb * nrhs);
    launch_source_gauss(src->p, vh * 12 * nrhs, 12345, stream());
    launch_spinor_from_aos(precision, src->p, vh * 192, vec(a->p, (long)fb), vh, nrhs, stream());
    launch_spinor_from_aos(precision, src->p, vh * 192, vec(b->p, (long)fb), vh, nrhs, stream());
    Vec va = vec(a->p, (long)fb), vb = vec(b->p, (long)fb);
    for (int w = 0; w < 3; ++w)
      hop(g, precision, recon, EPI_PLAIN, w & 1, 0, -1.0, (w & 1) ? vb : va, (w & 1) ? va : vb, vec(nullptr), nullptr,
          1.0, nrhs, nullptr, stream());
    hipEvent_t e0, e1;
    QHIP(hipEventCreate(&e0));
    QHIP(hipEventCreate(&e1));
    QHIP(hipEventRecord(e0, stream()));
    for (int i = 0; i < iters; ++i)
      hop(g, precision, recon, EPI_PLAIN, i & 1, 0, -1.0, (i & 1) ? vb : va, (i & 1) ? va : vb, vec(nullptr), nullptr,
          1.0, nrhs, nullptr, stream());
    QHIP(hipEventRecord(e1, stream()));
    QHIP(hipEventSynchronize(e1));
    float t = 0.f;
    QHIP(hipEventElapsedTime(&t, e0, e1));
    QHIP(hipEventDestroy(e0));
    QHIP(hipEventDestroy(e1));
    QHIP(hipGetLastError());
    *ms = (double)t / iters;
  });
}

int qcuBenchLinkProduct(int mfma, long site_legs, int iters, double* ms, double* checksum) {
  return guarded([&] {
    ensure_init();
    QREQ(ms && iters > 0, "qcuBenchLinkProduct: bad argument");
    QREQ(mfma == 0 || mfma == 1, "mfma must be 0 or 1");
    QREQ(site_legs > 0 && site_legs % 262144 == 0, "site_legs must be a positive multiple of 262144");
    DevBuf* o = ctx().buf("linkprod", sizeof(double) * 262144);
    launch_linkprod(mfma, site_legs, static_cast<double*>(o->p), stream());
    hipEvent_t e0, e1;
    QHIP(hipEventCreate(&e0));
    QHIP(hipEventCreate(&e1));
    QHIP(hipEventRecord(e0, stream()));
    for (int i = 0; i < iters; ++i) launch_linkprod(mfma, site_legs, static_cast<double*>(o->p), stream());
    QHIP(hipEventRecord(e1, stream()));
    QHIP(hipEventSynchronize(e1));
    QHIP(hipGetLastError());
    float t = 0.f;
    QHIP(hipEventElapsedTime(&t, e0, e1));
    QHIP(hipEventDestroy(e0));
    QHIP(hipEventDestroy(e1));
    *ms = (double)t / iters;
    if (checksum) {
      std::vector<double> h(262144);
      QHIP(hipMemcpy(h.data(), o->p, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
      double sum = 0.0;
      for (double v : h) sum += v;
      *checksum = sum;
    }
  });
}

int qcuBenchCopy(size_t bytes, int iters, double* ms) {
  return guarded([&] {
    ensure_init();
    QREQ(ms && iters > 0 && bytes > 0, "qcuBenchCopy: bad argument");
    DevBuf* a = ctx().buf("copy_a", bytes);
    DevBuf* b = ctx().buf("copy_b", bytes);
    QREQ(bytes % 16 == 0, "qcuBenchCopy: bytes must be a multiple of 16");
    QHIP(hipMemsetAsync(a->p, 1, bytes, stream()));
    launch_copy(b->p, a->p, bytes, stream());
    hipEvent_t e0, e1;
    QHIP(hipEventCreate(&e0));
    QHIP(hipEventCreate(&e1));
    QHIP(hipEventRecord(e0, stream()));
    for (int i = 0; i < iters; ++i) launch_copy((i & 1) ? a->p : b->p, (i & 1) ? b->p : a->p, bytes, stream());
    QHIP(hipEventRecord(e1, stream()));
    QHIP(hipEventSynchronize(e1));
    float t = 0.f;
    QHIP(hipEventElapsedTime(&t, e0, e1));
    QHIP(hipEventDestroy(e0));
    QHIP(hipEventDestroy(e1));
    *ms = (double)t / iters;
  });
}

}  // extern "C"
