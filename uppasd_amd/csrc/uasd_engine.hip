// uasd_engine.hip -- context, uploads and the C-ABI of libuasd_hip.so.
//
// A context mirrors the state the reference keeps in module arrays (ham_t,
// MomentData, FieldData, the LLG inputs) on one device, in the layout
// described in uasd_kernels.hpp.  Uploads convert the Fortran layout
// (3,Natom,Mensemble) to quads {x, y, z, w} indexed site*M+ens (w = mmom for
// spins) and compress the per-site coupling rows of ham%ncoup / ham%dm_vect /
// the anisotropy arrays to their distinct rows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/uasd_hip.h"
#include "uasd_launch.hpp"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                                  \
  do {                                                                                 \
    hipError_t _e = (expr);                                                            \
    if (_e != hipSuccess)                                                              \
      return fail(_e == hipErrorOutOfMemory ? UASD_ERR_NOMEM : UASD_ERR_HIP,          \
                  std::string(#expr) + ": " + hipGetErrorString(_e));                  \
  } while (0)

// Owned device allocation.
struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);  // teardown: no caller to report to
    p = nullptr;
    bytes = 0;
  }
  hipError_t ensure(size_t n) {
    if (n <= bytes && p) return hipSuccess;
    release();
    if (n == 0) return hipSuccess;
    hipError_t e = hipMalloc(&p, n);
    if (e == hipSuccess) bytes = n;
    else p = nullptr;
    return e;
  }
  template <typename T>
  T *as() const { return static_cast<T *>(p); }
};

// Owned pinned host memory, which kernels read and write in place.
struct PinBuf {
  void *p = nullptr;
  size_t bytes = 0;
  PinBuf() = default;
  PinBuf(const PinBuf &) = delete;
  PinBuf &operator=(const PinBuf &) = delete;
  ~PinBuf() {
    if (p) (void)hipHostFree(p);  // teardown: no caller to report to
  }
  hipError_t ensure(size_t n) {
    if (n <= bytes) return hipSuccess;
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
    const hipError_t e = hipHostMalloc(&p, n, hipHostMallocDefault);
    if (e == hipSuccess) bytes = n;
    else p = nullptr;
    return e;
  }
};

// Hash of a byte string (FNV-1a) for deduplicating rows.
struct RowKey {
  std::string bytes;
  bool operator==(const RowKey &o) const { return bytes == o.bytes; }
};
struct RowKeyHash {
  size_t operator()(const RowKey &k) const {
    uint64_t h = 1469598103934665603ULL;
    for (unsigned char c : k.bytes) h = (h ^ c) * 1099511628211ULL;
    return (size_t)h;
  }
};

struct Timing {
  int64_t launches = 0;
  double ms = 0.0;
};

// Fixed device scratch of uasd_energy_terms_noalloc: partial sums per
// (chunk, ensemble) and the sums per (segment, ensemble), 4 doubles each.
constexpr size_t kScratchDoubles = (size_t)1 << 19;  // 4 MiB per device
constexpr int kMaxDevices = 64;

}  // namespace

// One copy per device, held until the process ends.  On the host the name is
// only a stand-in for the symbol: kernels and copies take the device address
// that scratch_init looks up, never `scratch` itself.
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {

std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

// Device address of `device`'s copy of the scratch array, looked up once per
// device; the caller has made `device` current.
int scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices)
    return fail(UASD_ERR_UNSUPPORTED, "device index beyond the scratch table (64 devices)");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return UASD_OK;
  void *p = nullptr;
  HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) return fail(UASD_ERR_HIP, "hipGetSymbolAddress returned a null scratch address");
  g_scratch_ptr[device] = static_cast<double *>(p);
  return UASD_OK;
}

double *scratch_of(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[device];
}

}  // namespace

// ----------------------------------------------------------------- context
struct uasd_ctx {
  int N = 0, M = 0, prec = UASD_FP64, device = 0;
  // device site order: slot d holds reference site site_of(d) (see HamDev)
  int order_na = 1;
  int order_nc = 0;  // sites per basis atom (N when order_na = 1)
  hipStream_t own_stream = nullptr, stream = nullptr;
  size_t rsize = 8;  // sizeof(R)

  // host-side descriptors kept for class building / colouring
  int W = 0, ex_rows = 0;
  std::vector<int> ex_row_of_site;  // (N)
  std::vector<int> nbr_host;        // (W*N) slot-major, 0-based
  std::vector<int> ex_len_host;     // (ex_rows)
  bool ex_full = false;             // every exchange row holds W neighbours
  int Wd = 0, dm_rows = 0;
  std::vector<int> dm_row_of_site, dnbr_host, dm_len_host;
  std::vector<int> an_row_of_site;
  int an_rows = 0;
  int ext_mode = 0;
  std::vector<double> ext_u_host;  // (3*M)

  // device buffers
  DevBuf nbr, ex_len, cpl;
  DevBuf dnbr, dm_len, dv;
  DevBuf nbr16, dnbr16;  // int16 index differences when they all fit (else empty)
  bool use16 = false, use16_dm = false;
  DevBuf an_type, an_vals;
  DevBuf cls, classes;
  DevBuf ext_u, ext_full;
  DevBuf spins;   // quad arrays: e, p, b2
  DevBuf field;   // beff quads for the unfused path
  DevBuf scratch; // emomM quads (w = 1) for host field calls
  DevBuf hostio;  // host arrays on their way in or out (upload_vec, download_vec)
  PinBuf pinio;   // the same for small arrays
  PinBuf pinsum;  // final sums of a few (segment, ensemble) pairs
  DevBuf noise;   // injected N(0,1) quads
  DevBuf nsave;   // fused steps: deviates drawn by the predictor for the corrector
  DevBuf llgarr;  // lambda, temp, lande (double, N each)
  DevBuf energy;  // per q energy terms
  DevBuf partial, redout;
  DevBuf mcbuf;   // per-ensemble delta/beta/hbeta/ext + colour site lists

  bool have_ex = false, have_state = false, have_llg = false;
  bool classes_dirty = true;
  bool dm_shared = false;  // DM bonds = exchange bonds at every site (fused gather)
  bool tune_no_fuse = false;  // keep the separate DM gather (a tuning choice)

  // LLG parameters
  double dt = 1e-16, temprescale = 1.0, bn = 1.0;
  double lam0 = 0, temp0 = 0, lande0 = 1;
  bool lam_uniform = true, temp_uniform = true, lande_uniform = true;
  bool m_uniform = false;  // every moment magnitude equal (m0), as uploaded
  double m0 = 0;
  int noise_mode = UASD_NOISE_NONE;
  uint64_t seed = 0;
  uint64_t step = 0;      // LLG step counter (Philox counter)
  uint64_t mc_sweep = 0;  // MC sweep counter

  // launch shapes of the gathering kernels: 0 fused LLG, 1 field, 2 MC
  uasd::Tune tune[3];

  // lattice dimensions (reference site i = b + NA*(x + N1*(y + N2*z))) and
  // the translation-invariant stencil of the lists, when there is one
  int lat_na = 0, lat_n1 = 0, lat_n2 = 0, lat_n3 = 0;
  int64_t lds_max = 64 * 1024;  // LDS one workgroup may use (opt-in maximum)
  struct Stencil {
    bool ok = false;
    int W = 0, rx = 0, ry = 0, rz = 0;
    std::vector<int> bp, dx, dy, dz;  // (NA*W)
  } st_ex, st_dm;
  bool stencil_ok = false, stencil_dirty = true;
  DevBuf tile_off;
  int tile_off_shape = 0;
  std::vector<int> cls_host;       // site class per device slot
  bool one_class = false;          // every site is of class class0
  uasd::SiteClass class0{0, -1, -1, 0};
  int64_t cls_version = 0;         // bumped by every class rebuild
  int64_t ucls_version = -1;       // cls_version the per-basis check below is for
  int ucls = 0, cls_b[8] = {0};

  // segments (replicas of a batch): site ranges, their chunks, accumulators
  int nseg = 0;
  std::vector<int> seg_off;  // (nseg+1)
  int nchunks = 0;
  DevBuf seg_dev;            // int2 chunks (nchunks), int seg_chunk (nseg+1), int seg_n (nseg)
  DevBuf seg_partial, seg_out, acc;
  int64_t acc_samples = 0;

  // step graphs: replayed for runs of graph_steps LLG steps / MC
  // sweeps; the Philox counters then live in ctr (0 LLG step, 1 MC sweep).
  int graph_steps = 0;
  uint64_t gen = 0;           // bumped whenever a recorded graph may be stale
  uint64_t graphs_gen = 0;
  DevBuf ctr;
  bool ctr_valid[2] = {false, false};
  uint64_t ctr_val[2] = {0, 0};
  uasd::Recording *rec = nullptr;  // while a graph of steps or sweeps is built
  bool replays_off = false;   // an automatic replay failed on this stream
  struct Graph {
    hipGraph_t g = nullptr;
    hipGraphExec_t exec = nullptr;
  };
  std::map<std::tuple<int, int, int, uint64_t>, Graph> graphs;  // kind, alg/mode, K, seed
  // steps or sweeps launched one by one under unchanged settings (see
  // repeats_pay): kind, alg/mode, seed -> gen, count
  std::map<std::tuple<int, int, uint64_t>, std::pair<uint64_t, int64_t>> repeats;

  // colouring
  int ncolors = 0;
  std::vector<int> color_of_site, color_ptr, color_sites;
  // per colour: its slots are color_start + i * color_stride (stride 0: not
  // an arithmetic progression, the kernels read color_sites)
  std::vector<int> color_start, color_stride;
  bool coloring_dirty = true;

  // the independent systems of the lattice and their tables for the resident
  // MC kernel (built with the first MC call after a Hamiltonian change)
  struct Resident {
    bool ok = false;
    int ncomp = 0, nmax = 0;
    int64_t waves = 0;  // of one ensemble: of a half step; of all colours of a sweep
    DevBuf buf;
    uasd::ResDev dev{};
    int64_t cls_version = -1;
    int64_t col_version = -1;
  } res, lres;  // for MC sweeps (colour order), for LLG steps (device order)
  int64_t col_version = 0;  // bumped by every colouring rebuild

  // launches by path (uasd_launch_counts)
  int64_t launches[UASD_NUM_LAUNCH_KINDS] = {};

  // Per-kernel timing: an event pair is recorded around each launch without
  // a host wait; pairs are resolved when the totals are read.
  bool timing = false;
  int timing_every = 1;       // time one launch in timing_every of each kind
  bool timing_region = false; // time every uasd_sd_steps / uasd_mc_sweeps call (kind 6)
  int64_t timing_tick[7] = {};
  Timing timers[7];  // 0 predictor, 1 corrector, 2 field, 3 MC, 4 LLG graph, 5 MC graph, 6 call
  hipEvent_t region_cur = nullptr;
  std::vector<hipEvent_t> ev_pool;  // free events
  struct Pending {
    hipEvent_t a, b;
    int kind;
  };
  std::vector<Pending> pending;
  hipEvent_t cur = nullptr;
};

void build_stencil(uasd_ctx *c);
bool tile_fits(const uasd_ctx *c, int k);
int make_tile(uasd_ctx *c, int k, uasd::TileDev &t);

namespace {

void destroy_graphs(uasd_ctx *c);
int sd_steps_run(uasd_ctx *c, int alg, int64_t nsteps);
int llg_steps(uasd_ctx *c, int alg, int64_t n, bool in_graph);
int mc_sweeps_run(uasd_ctx *c, char mode, const uasd::MCParams &mp, int64_t nsweeps,
                  uint64_t seed);

// Reference site held by device slot d, and the slot of reference site i.
inline int site_of(const uasd_ctx *c, int d) {
  return c->order_na == 1 ? d : (d % c->order_nc) * c->order_na + d / c->order_nc;
}
inline int slot_of(const uasd_ctx *c, int i) {
  return c->order_na == 1 ? i : (i % c->order_na) * c->order_nc + i / c->order_na;
}

// Bits that hold the basis shift in an int16 list entry.
int idx_kb(const uasd_ctx *c) {
  int kb = 0;
  while ((1 << kb) < c->order_na) ++kb;
  return kb;
}


// Quad buffers: one Quad<R> = {x, y, z, w} per q = site*M + ens.
size_t quad_bytes(const uasd_ctx *c) { return (size_t)c->N * c->M * 4 * c->rsize; }

// spins holds three quad arrays: 0 e (emom, w = mmom), 1 p (emom2, w = mmom),
// 2 b2 (b2eff, w unused).
template <typename R>
uasd::Quad<R> *quads(const uasd_ctx *c, const DevBuf &b, int k = 0) {
  return reinterpret_cast<uasd::Quad<R> *>(static_cast<char *>(b.p) + (size_t)k * quad_bytes(c));
}

template <typename R>
uasd::HamDev<R> ham_view(const uasd_ctx *c) {
  uasd::HamDev<R> h{};
  h.N = c->N;
  h.M = c->M;
  h.mdiv = uasd::make_fast_div((uint32_t)c->M);
  h.W = c->W;
  h.ex_rows = c->ex_rows;
  h.ex_full = c->ex_full ? 1 : 0;
  h.nbr = c->nbr.as<int>();
  h.nbr16 = c->use16 ? c->nbr16.as<int16_t>() : nullptr;
  h.ex_len = c->ex_len.as<int>();
  h.cpl = c->cpl.as<R>();
  h.Wd = c->Wd;
  h.dm_rows = c->dm_rows;
  h.dnbr = c->dnbr.as<int>();
  h.dnbr16 = c->use16_dm ? c->dnbr16.as<int16_t>() : nullptr;
  h.dm_len = c->dm_len.as<int>();
  h.dm_shared = c->dm_shared && !c->tune_no_fuse ? 1 : 0;
  if (c->Wd > 0) {
    size_t n = (size_t)c->Wd * c->dm_rows;
    h.dvx = c->dv.as<R>();
    h.dvy = h.dvx + n;
    h.dvz = h.dvy + n;
  }
  if (c->an_rows > 0) {
    h.an_type = c->an_type.as<int>();
    const R *v = c->an_vals.as<R>();
    size_t n = (size_t)c->an_rows;
    h.an_ex = v;
    h.an_ey = v + n;
    h.an_ez = v + 2 * n;
    h.an_k1 = v + 3 * n;
    h.an_k2 = v + 4 * n;
    h.an_sb = v + 5 * n;
  }
  h.cls = c->cls.as<int>();
  h.classes = c->classes.as<uasd::SiteClass>();
  // Scalar couplings take a load per neighbour off the texture-address units,
  // which bound a full chip (film of 262,144 sites, Depondt FP64 25.2 -> 20.6
  // us a step; 170,368 sites with 14 neighbours 25.6 -> 23.3), but each batch
  // waits for them on top of its gathers, which a chip that is mostly waiting
  // anyway feels (16,000 sites with 58 neighbours 16.5 -> 17.4).
  h.one = !c->one_class ? 0 : (int64_t)c->N * c->M > 131072 ? 2 : 1;
  h.c0 = c->class0;
  h.ext_mode = c->ext_mode;
  h.order_na = c->order_na;
  h.idx_kb = idx_kb(c);
  h.order_nc = c->order_na == 1 ? c->N : c->order_nc;
  h.ext_u = c->ext_u.as<R>();
  if (c->ext_mode == 2) h.ext_q = quads<R>(c, c->ext_full);
  return h;
}

template <typename R>
int upload_converted(hipStream_t s, DevBuf &dst, const std::vector<double> &src) {
  std::vector<R> tmp(src.begin(), src.end());
  HIP_TRY(dst.ensure(std::max<size_t>(1, tmp.size()) * sizeof(R)));
  if (!tmp.empty())
    HIP_TRY(hipMemcpyAsync(dst.p, tmp.data(), tmp.size() * sizeof(R), hipMemcpyHostToDevice, s));
  HIP_TRY(hipStreamSynchronize(s));
  return UASD_OK;
}

int upload_real(uasd_ctx *c, DevBuf &dst, const std::vector<double> &src) {
  return c->prec == UASD_FP64 ? upload_converted<double>(c->stream, dst, src)
                              : upload_converted<float>(c->stream, dst, src);
}

template <typename T>
int upload_raw(uasd_ctx *c, DevBuf &dst, const std::vector<T> &src) {
  HIP_TRY(dst.ensure(std::max<size_t>(1, src.size()) * sizeof(T)));
  if (!src.empty())
    HIP_TRY(hipMemcpyAsync(dst.p, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice,
                           c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  return UASD_OK;
}

// Host (3,N,M) Fortran arrays cross as they are and are turned into quads, or
// made from them, by a kernel: p = i + N*k is the pair of reference site i and
// ensemble k, q its quad in device order.  A transfer's bound is then the copy
// itself; the host threads convert nothing.  Arrays pass through a device
// buffer of at most kIoPairs pairs, in stream order.  Against conversion on a
// host thread with pageable quads in between: a step of the host-array halves
// at 65,536 spins 2.13 -> 1.55 ms, moments of 4.1e6 pairs read back 95 -> 34 ms.
// A device with no room for that takes them in smaller pieces (io_pairs).
constexpr size_t kIoPairs = (size_t)1 << 22, kIoPairsLeast = (size_t)1 << 16;

// Host bytes of one pair in uasd_set_moments, its direction and magnitude, and
// the bytes of b2eff they pass through: its quads, which in FP32 hold half of
// the pairs at a time, or all of up to 65,536 (a second pair of copies is 9 us).
constexpr size_t kRawMoment = 4 * sizeof(double);
size_t raw_room(const uasd_ctx *c) {
  const size_t pairs = (size_t)c->N * c->M;
  return std::max(quad_bytes(c), kRawMoment * std::min<size_t>(pairs, 65536));
}

// the w of the quads an upload writes
struct PackW {
  int from_state = 0;  // 1: the moment magnitudes of the state's quads
  double value = 0.0;  // else this constant
};

// In device order, the quad of reference site i, ensemble k.
struct PairMap {
  int M, na, nc;
  uasd::FastDiv ndiv;  // division by N
  int N;
  __device__ __forceinline__ size_t quad(size_t p) const {
    const uint32_t k = uasd::fast_div((uint32_t)p, ndiv), i = (uint32_t)p - k * (uint32_t)N;
    const uint32_t d = na == 1 ? i : (i % na) * (uint32_t)nc + i / na;
    return (size_t)d * M + k;
  }
};

// Pairs [p0, p0 + n) of a staged array a (and w) into their quads.  wsrc and
// dst may be the same array: each thread reads and writes its own quad.
// dst2, where given, gets the same quads.
template <typename R>
__global__ void __launch_bounds__(256)
    k_pack(PairMap m, size_t p0, size_t n, const double *__restrict__ a,
           const double *__restrict__ w, const uasd::Quad<R> *wsrc, double wconst,
           uasd::Quad<R> *dst, uasd::Quad<R> *dst2) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const size_t q = m.quad(p0 + t);
  const uasd::Quad<R> v{(R)a[3 * t], (R)a[3 * t + 1], (R)a[3 * t + 2],
                        w ? (R)w[t] : wsrc ? wsrc[q].w : (R)wconst};
  dst[q] = v;
  if (dst2) dst2[q] = v;
}

// The reverse: xyz, or xyz*w (emomM), of pairs [p0, p0 + n) in FP64.
template <typename R>
__global__ void __launch_bounds__(256)
    k_unpack(PairMap m, size_t p0, size_t n, const uasd::Quad<R> *__restrict__ src, int times_w,
             double *__restrict__ out) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const uasd::Quad<R> v = src[m.quad(p0 + t)];
  const double w = times_w ? (double)v.w : 1.0;
  out[3 * t] = (double)v.x * w;
  out[3 * t + 1] = (double)v.y * w;
  out[3 * t + 2] = (double)v.z * w;
}

PairMap pair_map(const uasd_ctx *c) {
  return PairMap{c->M, c->order_na, c->order_na == 1 ? c->N : c->order_nc,
                 uasd::make_fast_div((uint32_t)c->N), c->N};
}

// The host arrays of one call.  Large ones are copied through the context's
// device buffer.  Small ones (kPinPairs) go through pinned memory that the
// kernels read and write in place: a copy command of up to 400 KB costs more
// than the conversion kernel it would feed.  Copies against pinned memory, us a
// call (moments read back; a step of the host-array halves): 54 sites 39 -> 17,
// 255 -> 139; 4056 sites 55 -> 25, 384 -> 189; 16,000 sites 83 -> 51, 540 -> 334.
// The first call pins room for the arrays of any call in about 10 us; pinning
// what each call needs had the larger ones free and pin again (first halves of a
// step at 8192 sites 330 -> 1010 us).  wait() ends the call's transfers; a call
// that ends early waits before its caller gets the arrays back.
struct HostIo {
  static constexpr size_t kPinPairs = 16384, kPinArrays = 8;
  uasd_ctx *c;
  bool open = false;
  size_t used = 0;  // doubles of c->pinio in use
  struct Out {
    double *to;
    const double *from;
    size_t n;
  };
  std::vector<Out> outs;
  explicit HostIo(uasd_ctx *cc) : c(cc) {}
  ~HostIo() {
    if (open) (void)hipStreamSynchronize(c->stream);  // the call's own error is reported
  }
  bool small() const { return (size_t)c->N * c->M <= kPinPairs; }
  // n doubles of pinned memory that stay untouched until wait()
  int pinned(size_t n, double **p) {
    HIP_TRY(c->pinio.ensure(kPinArrays * 3 * (size_t)c->N * c->M * sizeof(double)));
    if ((used + n) * sizeof(double) > c->pinio.bytes)
      return fail(UASD_ERR_STATE, "pinned staging exhausted");
    *p = static_cast<double *>(c->pinio.p) + used;
    used += n;
    return UASD_OK;
  }
  int wait() {
    open = false;
    HIP_TRY(hipStreamSynchronize(c->stream));
    for (const Out &o : outs) std::memcpy(o.to, o.from, o.n * sizeof(double));
    outs.clear();
    used = 0;
    return UASD_OK;
  }
};

int launch_pack(uasd_ctx *c, DevBuf &b, int k, size_t p0, size_t n, const double *a,
                const double *w, const PackW &pw, bool twice = false) {
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  if (c->prec == UASD_FP64)
    hipLaunchKernelGGL(k_pack<double>, grid, block, 0, c->stream, pair_map(c), p0, n, a, w,
                       pw.from_state ? quads<double>(c, c->spins, 0) : nullptr, pw.value,
                       quads<double>(c, b, k), twice ? quads<double>(c, b, k + 1) : nullptr);
  else
    hipLaunchKernelGGL(k_pack<float>, grid, block, 0, c->stream, pair_map(c), p0, n, a, w,
                       pw.from_state ? quads<float>(c, c->spins, 0) : nullptr, pw.value,
                       quads<float>(c, b, k), twice ? quads<float>(c, b, k + 1) : nullptr);
  HIP_TRY(hipGetLastError());
  return UASD_OK;
}

int launch_unpack(uasd_ctx *c, const DevBuf &b, int k, size_t p0, size_t n, bool times_w,
                  double *out) {
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  if (c->prec == UASD_FP64)
    hipLaunchKernelGGL(k_unpack<double>, grid, block, 0, c->stream, pair_map(c), p0, n,
                       quads<double>(c, b, k), times_w ? 1 : 0, out);
  else
    hipLaunchKernelGGL(k_unpack<float>, grid, block, 0, c->stream, pair_map(c), p0, n,
                       quads<float>(c, b, k), times_w ? 1 : 0, out);
  HIP_TRY(hipGetLastError());
  return UASD_OK;
}

// Pairs that pass through c->hostio at a time, allocated with the first call.
int io_pairs(uasd_ctx *c, size_t *pairs) {
  constexpr size_t kBytes = 3 * sizeof(double);
  *pairs = std::min((size_t)c->N * c->M, kIoPairs);
  while (!c->hostio.p) {
    const hipError_t e = c->hostio.ensure(*pairs * kBytes);
    if (e == hipSuccess) break;
    if (e != hipErrorOutOfMemory || *pairs <= kIoPairsLeast) HIP_TRY(e);
    (void)hipGetLastError();  // the smaller piece's launches have errors of their own
    *pairs = std::max(*pairs / 4, kIoPairsLeast);
  }
  *pairs = std::min(*pairs, c->hostio.bytes / kBytes);
  return UASD_OK;
}

// Host array a into quad array k of buffer b.  Asynchronous: a must stay as it
// is until io.wait().
int upload_vec(HostIo &io, DevBuf &b, int k, const double *a, PackW w) {
  uasd_ctx *c = io.c;
  HIP_TRY(b.ensure(std::max(b.bytes, (size_t)(k + 1) * quad_bytes(c))));
  const size_t total = (size_t)c->N * c->M;
  io.open = true;
  if (io.small()) {
    double *sa = nullptr;
    if (int r = io.pinned(3 * total, &sa)) return r;
    std::memcpy(sa, a, 3 * total * sizeof(double));
    return launch_pack(c, b, k, 0, total, sa, nullptr, w);
  }
  size_t step = 0;
  if (int r = io_pairs(c, &step)) return r;
  double *sa = c->hostio.as<double>();
  for (size_t p0 = 0; p0 < total; p0 += step) {
    const size_t n = std::min(step, total - p0);
    HIP_TRY(hipMemcpyAsync(sa, a + 3 * p0, 3 * n * sizeof(double), hipMemcpyHostToDevice,
                           c->stream));
    if (int r = launch_pack(c, b, k, p0, n, sa, nullptr, w)) return r;
  }
  return UASD_OK;
}

// Quad array k of buffer b into host array out (times_w: emomM = xyz*w).
// Asynchronous: out is complete after io.wait().
int download_vec(HostIo &io, const DevBuf &b, int k, double *out, bool times_w) {
  uasd_ctx *c = io.c;
  const size_t total = (size_t)c->N * c->M;
  io.open = true;
  if (io.small()) {
    double *so = nullptr;
    if (int r = io.pinned(3 * total, &so)) return r;
    io.outs.push_back({out, so, 3 * total});
    return launch_unpack(c, b, k, 0, total, times_w, so);
  }
  size_t step = 0;
  if (int r = io_pairs(c, &step)) return r;
  double *so = c->hostio.as<double>();
  for (size_t p0 = 0; p0 < total; p0 += step) {
    const size_t n = std::min(step, total - p0);
    if (int r = launch_unpack(c, b, k, p0, n, times_w, so)) return r;
    HIP_TRY(hipMemcpyAsync(out + 3 * p0, so, 3 * n * sizeof(double), hipMemcpyDeviceToHost,
                           c->stream));
  }
  return UASD_OK;
}

// Whether every site's DM neighbours are its exchange neighbours, in the same
// order and number, at most kFusedW of them (or there is no DM term): the
// field kernels then gather each neighbour once for both sums.
bool dm_lists_shared(const uasd_ctx *c) {
  if (c->Wd == 0 || c->dm_row_of_site.empty()) return false;
  if (c->W > uasd::kFusedW) return false;
  const int N = c->N;
  for (int i = 0; i < N; ++i) {
    const int dr = c->dm_row_of_site[i];
    if (dr < 0) continue;
    const int er = c->ex_row_of_site.empty() ? 0 : c->ex_row_of_site[i];
    const int L = c->ex_len_host[er];
    if (c->dm_len_host[dr] != L) return false;
    for (int j = 0; j < L; ++j)
      if (c->dnbr_host[(size_t)j * N + i] != c->nbr_host[(size_t)j * N + i]) return false;
  }
  return true;
}

// may_alloc = false: fail rather than grow the device tables (the no-alloc
// entry point), i.e. when the class tables outgrow the buffers of the last
// build.
int rebuild_classes(uasd_ctx *c, bool may_alloc = true) {
  if (!c->classes_dirty) return UASD_OK;
  std::map<std::tuple<int, int, int>, int> ids;
  std::vector<int> cls(c->N);
  std::vector<uasd::SiteClass> table;
  for (int i = 0; i < c->N; ++i) {
    int er = c->ex_row_of_site.empty() ? 0 : c->ex_row_of_site[i];
    int dr = c->dm_row_of_site.empty() ? -1 : c->dm_row_of_site[i];
    int ar = c->an_row_of_site.empty() ? -1 : c->an_row_of_site[i];
    auto key = std::make_tuple(er, dr, ar);
    auto it = ids.find(key);
    if (it == ids.end()) {
      it = ids.emplace(key, (int)table.size()).first;
      table.push_back(uasd::SiteClass{er, dr, ar, 0});
    }
    cls[i] = it->second;
  }
  c->dm_shared = dm_lists_shared(c);
  if (!may_alloc && (!c->cls.p || !c->classes.p || c->cls.bytes < cls.size() * sizeof(int) ||
                     c->classes.bytes < table.size() * sizeof(uasd::SiteClass)))
    return fail(UASD_ERR_STATE,
                "the site-class tables are not on the device yet; call uasd_energy_terms (or "
                "any field, step or sweep entry point) once after the last Hamiltonian upload");
  int r = upload_raw(c, c->cls, cls);
  if (r) return r;
  r = upload_raw(c, c->classes, table);
  if (r) return r;
  c->cls_host = cls;
  c->one_class = table.size() == 1;
  c->class0 = table[0];
  c->cls_version += 1;
  c->classes_dirty = false;
  c->gen += 1;
  return UASD_OK;
}

// Distinct rows of a per-site table.  row_ref[i] is the Hamiltonian row of
// site i; `len` and `vals(width*hdim)` describe that row.
struct RowSet {
  std::vector<int> row_of_site;
  std::vector<int> len;
  std::vector<std::vector<double>> vals;
};

RowSet dedupe_rows(int N, const std::vector<int> &row_ref, const int *lenarr, const double *vals,
                   int width, int hdim) {
  RowSet rs;
  rs.row_of_site.resize(N);
  std::unordered_map<int, int> by_ref;  // Hamiltonian row -> distinct row
  std::unordered_map<RowKey, int, RowKeyHash> by_content;
  for (int i = 0; i < N; ++i) {
    int ref = row_ref[i];
    auto f = by_ref.find(ref);
    if (f != by_ref.end()) {
      rs.row_of_site[i] = f->second;
      continue;
    }
    int L = lenarr[ref];
    RowKey key;
    key.bytes.assign(reinterpret_cast<const char *>(&L), sizeof(int));
    const double *v = vals + (size_t)ref * width * hdim;
    key.bytes.append(reinterpret_cast<const char *>(v), sizeof(double) * (size_t)L * hdim);
    auto g = by_content.find(key);
    int id;
    if (g == by_content.end()) {
      id = (int)rs.len.size();
      by_content.emplace(std::move(key), id);
      rs.len.push_back(L);
      rs.vals.emplace_back(v, v + (size_t)L * hdim);
    } else {
      id = g->second;
    }
    by_ref.emplace(ref, id);
    rs.row_of_site[i] = id;
  }
  return rs;
}

int check_ctx(uasd_ctx *c) {
  if (!c) return fail(UASD_ERR_ARG, "null context");
  return UASD_OK;
}

hipEvent_t take_event(uasd_ctx *c) {
  if (!c->ev_pool.empty()) {
    hipEvent_t e = c->ev_pool.back();
    c->ev_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

void tic(uasd_ctx *c, int kind) {
  if (!c->timing || c->rec) return;
  if (c->timing_tick[kind]++ % c->timing_every != 0) return;
  c->cur = take_event(c);
  // a start event that could not be recorded times nothing: back to the pool
  if (c->cur && hipEventRecord(c->cur, c->stream) != hipSuccess) {
    c->ev_pool.push_back(c->cur);
    c->cur = nullptr;
  }
}

int toc(uasd_ctx *c, int kind) {
  if (!c->timing || c->rec || !c->cur) return UASD_OK;
  hipEvent_t b = take_event(c);
  if (!b) return fail(UASD_ERR_HIP, "hipEventCreate failed");
  HIP_TRY(hipEventRecord(b, c->stream));
  c->pending.push_back({c->cur, b, kind});
  c->cur = nullptr;
  return UASD_OK;
}

// Event pair around a whole stepping call (kind 6), on the context stream.
int region_tic(uasd_ctx *c) {
  if (!c->timing_region || c->rec) return UASD_OK;
  c->region_cur = take_event(c);
  if (!c->region_cur) return fail(UASD_ERR_HIP, "hipEventCreate failed");
  const hipError_t err = hipEventRecord(c->region_cur, c->stream);
  if (err != hipSuccess) {  // no region opened: the event goes back to the pool
    c->ev_pool.push_back(c->region_cur);
    c->region_cur = nullptr;
  }
  HIP_TRY(err);
  return UASD_OK;
}

int region_toc(uasd_ctx *c) {
  if (!c->region_cur) return UASD_OK;
  hipEvent_t b = take_event(c);
  if (!b) return fail(UASD_ERR_HIP, "hipEventCreate failed");
  HIP_TRY(hipEventRecord(b, c->stream));
  c->pending.push_back({c->region_cur, b, 6});
  c->region_cur = nullptr;
  return UASD_OK;
}

// Where the launches of steps and sweeps go.
uasd::Queue queue(const uasd_ctx *c) { return {c->stream, c->rec}; }

// One launch of `kind` that runs now (not one recorded into a graph).
void count(uasd_ctx *c, int kind) {
  if (!c->rec) c->launches[kind] += 1;
}

int resolve_timing(uasd_ctx *c) {
  for (auto &p : c->pending) {
    HIP_TRY(hipEventSynchronize(p.b));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, p.a, p.b));
    c->timers[p.kind].launches += 1;
    c->timers[p.kind].ms += ms;
    c->ev_pool.push_back(p.a);
    c->ev_pool.push_back(p.b);
  }
  c->pending.clear();
  return UASD_OK;
}

template <typename R>
uasd::LLGDev<R> llg_view(uasd_ctx *c) {
  uasd::LLGDev<R> p{};
  const double *arr = c->llgarr.as<double>();
  p.lam = c->lam_uniform ? nullptr : arr;
  p.temp = c->temp_uniform ? nullptr : arr + c->N;
  p.lande = c->lande_uniform ? nullptr : arr + 2 * (size_t)c->N;
  p.lam0 = c->lam0;
  p.temp0 = c->temp0;
  p.lande0 = c->lande0;
  p.dt = c->dt;
  p.temprescale = c->temprescale;
  p.bn = c->bn;
  p.noise_mode = c->noise_mode;
  // a uniform T = 0 scales every deviate by zero: draw none
  if (c->temp_uniform && c->temp0 == 0.0 && p.noise_mode == UASD_NOISE_PHILOX)
    p.noise_mode = UASD_NOISE_NONE;
  p.seed = c->seed;
  p.step = c->step;
  if (c->noise_mode == UASD_NOISE_INJECTED) p.noise = quads<R>(c, c->noise);
  p.lc0 = uasd::lam_const<R>(c->lam0, c->dt, c->bn);
  if (c->lam_uniform && c->temp_uniform && c->m_uniform) {
    const double m = (double)(R)c->m0;  // as the kernels read it from the quads
    p.sig_uniform = 1;
    p.sigk0 = uasd::midpoint_sigma<R>(p.lc0.Dk, m, c->temp0, c->temprescale);
    p.sigp0 = uasd::depondt_sigma<R>(p.lc0.Dp, m, c->temp0, c->temprescale);
    p.sigh0 = uasd::heun_sigma<R>(p.lc0.Dh, m, c->temp0, c->temprescale, c->dt);
  }
  return p;
}

// Whether some bond spans `sites` slots or more, so that its system has more
// sites than that.  In a periodic crystal that is larger the first site's does.
bool bond_spans(const uasd_ctx *c, int sites) {
  auto spans = [&](const std::vector<int> &row, const std::vector<int> &len,
                   const std::vector<int> &list) {
    for (int i = 0; i < c->N && !row.empty(); ++i)
      for (int j = 0; row[i] >= 0 && j < len[row[i]]; ++j)
        if (std::abs(list[(size_t)j * c->N + i] - i) >= sites) return true;
    return false;
  };
  return spans(c->ex_row_of_site, c->ex_len_host, c->nbr_host) ||
         (c->Wd > 0 && spans(c->dm_row_of_site, c->dm_len_host, c->dnbr_host));
}

// Contiguous ranges of device slots that no bond crosses, as first slots.
std::vector<int> independent_ranges(const uasd_ctx *c) {
  const int N = c->N;
  std::vector<int> reach(N);  // furthest slot bonded to slot i or to one before it
  auto add = [&](const std::vector<int> &row, const std::vector<int> &len,
                 const std::vector<int> &nb, int W) {
    if (W == 0 || row.empty()) return;
    for (int j = 0; j < W; ++j)
      for (int i = 0; i < N; ++i)
        if (j < len[row[i]]) {
          const int n = nb[(size_t)j * N + i];
          reach[std::min(i, n)] = std::max(reach[std::min(i, n)], std::max(i, n));
        }
  };
  for (int i = 0; i < N; ++i) reach[i] = i;
  add(c->ex_row_of_site, c->ex_len_host, c->nbr_host, c->W);
  add(c->dm_row_of_site, c->dm_len_host, c->dnbr_host, c->Wd);
  std::vector<int> off(1, 0);
  for (int i = 0, far = 0; i < N; ++i) {
    far = std::max(far, reach[i]);
    if (far == i) off.push_back(i + 1);
  }
  return off;
}

// Builds c->lres, the systems of the lattice for resident LLG steps, where
// they are small enough for them.  Lattices over kLlgResLattice sites are not
// looked through: their batches fill the chip with the other kernels.
constexpr int kLlgResSites = uasd::kResThreads, kLlgResLattice = 16384, kLlgResItems = 131072;

int build_llg_resident(uasd_ctx *c) {
  auto &r = c->lres;
  if (r.cls_version == c->cls_version) return UASD_OK;
  r.ok = false;
  r.cls_version = c->cls_version;
  const int N = c->N, W = c->W, Wd = c->Wd;
  if (N > kLlgResLattice) return UASD_OK;
  if (bond_spans(c, kLlgResSites)) return UASD_OK;
  const std::vector<int> off = independent_ranges(c);
  const int ncomp = (int)off.size() - 1;
  int nmax = 0;
  for (int k = 0; k < ncomp; ++k) nmax = std::max(nmax, off[k + 1] - off[k]);
  if (nmax > kLlgResSites || uasd::res_lds_llg(c->rsize, nmax) > (size_t)c->lds_max)
    return UASD_OK;
  std::vector<uint16_t> nb((size_t)(W + Wd) * N);
  for (int k = 0; k < ncomp; ++k)
    for (int i = off[k]; i < off[k + 1]; ++i) {
      for (int j = 0; j < W; ++j)
        nb[(size_t)j * N + i] = (uint16_t)(c->nbr_host[(size_t)j * N + i] - off[k]);
      for (int j = 0; j < Wd; ++j)
        nb[(size_t)(W + j) * N + i] = (uint16_t)(c->dnbr_host[(size_t)j * N + i] - off[k]);
    }
  std::vector<uasd::SiteClass> cls(N);
  for (int i = 0; i < N; ++i)
    cls[i] = uasd::SiteClass{c->ex_row_of_site.empty() ? 0 : c->ex_row_of_site[i],
                             c->dm_row_of_site.empty() ? -1 : c->dm_row_of_site[i],
                             c->an_row_of_site.empty() ? -1 : c->an_row_of_site[i], 0};
  std::vector<char> all(cls.size() * sizeof(cls[0]) + off.size() * sizeof(int) +
                        nb.size() * sizeof(uint16_t));
  const size_t ooff = cls.size() * sizeof(cls[0]), onb = ooff + off.size() * sizeof(int);
  std::memcpy(all.data(), cls.data(), ooff);
  std::memcpy(all.data() + ooff, off.data(), off.size() * sizeof(int));
  std::memcpy(all.data() + onb, nb.data(), nb.size() * sizeof(uint16_t));
  if (upload_raw(c, r.buf, all)) {  // no room for tables that the launched kernels do not need
    (void)hipGetLastError();
    return UASD_OK;
  }
  const char *base = r.buf.as<char>();
  r.dev = uasd::ResDev{};
  r.dev.ncomp = ncomp;
  r.dev.nmax = nmax;
  r.dev.off = reinterpret_cast<const int *>(base + ooff);
  r.dev.cls = reinterpret_cast<const uasd::SiteClass *>(base);
  r.dev.nbr = reinterpret_cast<const uint16_t *>(base + onb);
  r.dev.dnbr = r.dev.nbr + (size_t)W * N;
  r.ncomp = ncomp;
  r.nmax = nmax;
  r.waves = 0;
  for (int k = 0; k < ncomp; ++k)
    r.waves += uasd::res_waves(off[k + 1] - off[k], (nmax + 63) / 64);
  r.ok = true;
  return UASD_OK;
}

// Whether a call's LLG steps run in k_llg_resident: systems of at most one
// site per thread of its workgroup.  Per step, two launches -> resident, FP64
// (FP32), one ensemble: 128 sites, 14 neighbours 9.7 -> 3.6 us (10.6 -> 3.3),
// 432 sites 11.3 -> 5.0 (11.3 -> 3.8), Depondt 12.4 -> 5.8, 58 neighbours 22.8
// -> 11.3 (18.2 -> 7.5), SIB 17.1 -> 12.9; 64 ensembles of 432 sites 13.1 ->
// 6.5.  With 1024 sites the one CU is as slow as the launches (58 neighbours
// 22.5 -> 22.5, film 13.7 -> 13.9, SIB 17.4 -> 24.0).  Fewer than 2040 idle
// wavefronts in FP64 and 4000 in FP32: Depondt, launches against resident, sites
// x systems, idle wavefronts in brackets, 64 x 2048 (205) FP64 12.0 -> 10.9 us,
// FP32 8.0 -> 7.8; 250 x 520 (252) 21.0 -> 14.0, 15.6 -> 10.3; 100 x 1280 (760)
// 12.1 -> 10.7, 8.0 -> 8.0; 65 x 2016 (2189) 12.1 -> 13.9, 8.4 -> 8.5; 1 x 2048
// (2019) 5.6 -> 3.6, 5.7 -> 2.4; 4 x 4096 (3866) 6.9 -> 7.8, 6.4 -> 4.4; 16 x 8192
// (6349) 12.0 -> 17.8, 8.0 -> 11.4; 1 x 131,072 11.2 -> 167, 7.4 -> 86.
// Not while the kernels are timed one by one, graphs were asked for or a launch
// shape was: a shape is one of the kernels that the resident launch would take
// the place of.
bool llg_can_be_resident(const uasd_ctx *c) {
  return c->lres.ok && c->lres.cls_version == c->cls_version && c->graph_steps == 0 &&
         (int64_t)c->N * c->M <= kLlgResItems &&
         uasd::res_idle_waves(c->lres.waves * c->M, (int64_t)c->N * c->M, 0.9) <
             (c->prec == UASD_FP32 ? 4000 : 2040);
}

bool llg_use_resident(const uasd_ctx *c) {
  return llg_can_be_resident(c) && !c->timing && c->tune[0].chosen != uasd::kShapeAsked;
}

// Steps whose Philox deviates are drawn in one launch ahead of them.  FP64
// deviates are a third of a predictor's instructions and, while the lattice
// leaves CUs idle, of its time: midpoint and Depondt steps of 432 to 16,000
// sites with 14 or 58 neighbours gain 0.3-0.8 us of 11-18.  At 65,536 sites
// the extra pass over them costs what it saves, and FP32 deviates are too
// cheap to gain at any size.  The extra launch wants a group of at least
// kDrawGroup steps to repay it: Depondt with 14 neighbours, us a step drawn in
// the predictor, in groups of 2, 4, 6, 16: 686 sites 11.7, 12.4, 11.6, 11.3,
// 11.0; 16,000 sites 11.8, 12.6, 11.8, 11.6, 11.3; 32,500 sites 12.6, 13.5,
// 12.9, 12.7, 12.4.
constexpr int kDrawGroup = 6;

int steps_ahead(const uasd_ctx *c) {
  return c->prec == UASD_FP64 && (int64_t)c->N * c->M <= 32768 ? 16 : 1;
}

// Steps of a resident launch: as many as deviates of 2^18 items cover, 4 to 64.
int64_t resident_steps(const uasd_ctx *c) {
  return std::max<int64_t>(4, std::min<int64_t>(64, 262144 / ((int64_t)c->N * c->M)));
}

// Steps whose deviates c->nsave holds: the most that any path of this context
// draws at once, from its sizes alone.  The buffer then never moves, so steps
// that a caller captured into a graph of its own keep a valid address whatever
// runs between its replays.
int64_t nsave_steps(const uasd_ctx *c) {
  const bool res = c->N <= kLlgResLattice && (int64_t)c->N * c->M <= kLlgResItems;
  return std::max<int64_t>(steps_ahead(c), res ? resident_steps(c) : 1);
}

int ready_for_llg(uasd_ctx *c) {
  if (!c->have_ex) return fail(UASD_ERR_STATE, "exchange not set (uasd_set_exchange)");
  if (!c->have_state) return fail(UASD_ERR_STATE, "moments not set (uasd_set_moments)");
  if (!c->have_llg) return fail(UASD_ERR_STATE, "LLG parameters not set (uasd_set_llg)");
  if (c->noise_mode == UASD_NOISE_INJECTED && !c->noise.p)
    return fail(UASD_ERR_STATE, "injected noise selected but no normals uploaded");
  if (c->noise_mode == UASD_NOISE_PHILOX) {
    void *old = c->nsave.p;
    HIP_TRY(c->nsave.ensure((size_t)nsave_steps(c) * quad_bytes(c)));
    if (c->nsave.p != old) c->gen += 1;  // captured graphs hold the old address
  }
  return rebuild_classes(c);
}

// Quad arrays in c->spins: 0 e (emom), 1 p (emom2), 2 b2 (b2eff).
// step_off >= 0: inside a recorded graph, the step is *ctr[0] + step_off.
bool sde_supported(int alg) {
  return alg == UASD_SDE_MIDPOINT || alg == UASD_SDE_HEUN || alg == UASD_SDE_DEPONDT ||
         alg == UASD_SDE_SIB || alg == UASD_SDE_SPHMID;
}

// solvers that keep b2eff between the halves
bool sde_b2eff(int alg) { return alg == UASD_SDE_HEUN || alg == UASD_SDE_DEPONDT; }

// ahead >= 0: the step's deviates lie in quad array `ahead` of c->nsave.
template <typename R>
int run_llg_half(uasd_ctx *c, int alg, int half, bool fused, bool write_e,
                 int64_t step_off = -1, int ahead = -1) {
  uasd::HamDev<R> h = ham_view<R>(c);
  uasd::LLGDev<R> prm = llg_view<R>(c);
  if (step_off >= 0) {
    prm.step = (uint64_t)step_off;
    prm.step_dev = c->ctr.as<uint64_t>();
  }
  // a fused predictor/corrector pair draws the deviates once: the predictor
  // stores them, the corrector of the same step reads them back
  if (fused && prm.noise_mode == UASD_NOISE_PHILOX) {
    prm.nsave = quads<R>(c, c->nsave, std::max(ahead, 0));
    prm.nready = ahead >= 0 ? 1 : 0;
  }
  uasd::Quad<R> *e = quads<R>(c, c->spins, 0), *p = quads<R>(c, c->spins, 1),
                *b2 = quads<R>(c, c->spins, 2);
  const uasd::Quad<R> *beff = fused ? nullptr : quads<R>(c, c->field);
  uasd::Quad<R> *out = write_e ? e : p;
  if (fused && c->tune[0].tile > 0) {
    build_stencil(c);
    if (tile_fits(c, c->tune[0].tile)) {
      uasd::TileDev t;
      if (int r = make_tile(c, c->tune[0].tile, t)) return r;
      tic(c, half);
      HIP_TRY(uasd::launch_llg_tile<R>(queue(c), t, c->tune[0].pipe, alg, half, h, prm, e, p, b2,
                                       out));
      count(c, UASD_LAUNCH_LLG_TILE);
      return toc(c, half);
    }
  }
  tic(c, half);
  HIP_TRY(uasd::launch_llg<R>(queue(c),
                              uasd::default_tune(c->tune[0], (int64_t)c->N * c->M, c->W), alg,
                              half, fused, h, prm, e, p, b2, beff, out));
  count(c, UASD_LAUNCH_LLG_LIST);
  return toc(c, half);
}

// parts: also write beff1 and beff2 into quad arrays 1 and 2 of c->field;
// want_beff = false: the energy alone.
template <typename R>
int run_field(uasd_ctx *c, bool from_scratch, bool want_energy, bool parts = false,
              bool want_beff = true) {
  uasd::HamDev<R> h = ham_view<R>(c);
  const uasd::Quad<R> *src = from_scratch ? quads<R>(c, c->scratch) : quads<R>(c, c->spins, 0);
  HIP_TRY(c->field.ensure(std::max(c->field.bytes, (parts ? 3 : 1) * quad_bytes(c))));
  double *en = nullptr;
  if (want_energy) {
    HIP_TRY(c->energy.ensure((size_t)c->N * c->M * sizeof(double)));
    en = c->energy.as<double>();
  }
  tic(c, 2);
  HIP_TRY(uasd::launch_field<R>(c->stream,
                                uasd::default_tune(c->tune[1], (int64_t)c->N * c->M, c->W), h, src,
                                want_beff ? quads<R>(c, c->field) : nullptr, en,
                                parts ? quads<R>(c, c->field, 1) : nullptr));
  return toc(c, 2);
}

// Where a call's final sums are written: a few of them straight into pinned
// host memory (the call waits for the stream anyway, and saves a copy
// command), more into the device buffer d.  sums_back waits and brings them to
// `out`.
constexpr size_t kPinSums = 512;

int sums_out(uasd_ctx *c, DevBuf &d, size_t n, double **dst) {
  if (n <= kPinSums) {
    HIP_TRY(c->pinsum.ensure(kPinSums * sizeof(double)));
    *dst = static_cast<double *>(c->pinsum.p);
    return UASD_OK;
  }
  HIP_TRY(d.ensure(n * sizeof(double)));
  *dst = d.as<double>();
  return UASD_OK;
}

int sums_back(uasd_ctx *c, const double *src, size_t n, double *out) {
  const bool pinned = src == c->pinsum.p;
  if (!pinned)
    HIP_TRY(hipMemcpyAsync(out, src, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  if (pinned) std::memcpy(out, src, n * sizeof(double));
  return UASD_OK;
}

// FP64 sums per ensemble of emomM (and of the per-q energy terms written by
// the field kernel when with_energy).
template <typename R>
int reduce_moments(uasd_ctx *c, bool with_energy, bool from_scratch, std::vector<double> &out) {
  const int nv = with_energy ? 4 : 3;
  const int nblocks = std::max(1, std::min(1024, (c->N + 255) / 256));
  HIP_TRY(c->partial.ensure((size_t)c->M * nblocks * nv * sizeof(double)));
  const size_t nout = (size_t)c->M * nv;
  double *dst = nullptr;
  if (int r = sums_out(c, c->redout, nout, &dst)) return r;
  const uasd::Quad<R> *s = from_scratch ? quads<R>(c, c->scratch) : quads<R>(c, c->spins, 0);
  HIP_TRY(uasd::launch_reduce<R>(c->stream, c->N, c->M, s,
                                 with_energy ? c->energy.as<double>() : nullptr, nv,
                                 c->partial.as<double>(), nblocks, dst));
  out.resize(nout);
  return sums_back(c, dst, nout, out.data());
}

int build_coloring(uasd_ctx *c) {
  if (!c->coloring_dirty) return UASD_OK;
  const int N = c->N;
  // undirected bond graph from exchange and DM lists
  std::vector<std::vector<int>> adj(N);
  auto add_list = [&](const std::vector<int> &row_of_site, const std::vector<int> &len,
                      const std::vector<int> &nb, int W) {
    if (W == 0 || row_of_site.empty()) return;
    for (int i = 0; i < N; ++i) {
      int L = len[row_of_site[i]];
      for (int j = 0; j < L; ++j) {
        int n = nb[(size_t)j * N + i];
        if (n == i) continue;
        adj[i].push_back(n);
        adj[n].push_back(i);
      }
    }
  };
  add_list(c->ex_row_of_site, c->ex_len_host, c->nbr_host, c->W);
  add_list(c->dm_row_of_site, c->dm_len_host, c->dnbr_host, c->Wd);
  std::vector<int> col(N, -1);
  int ncol = 0;
  std::vector<int> mark;
  // greedy colouring visiting the sites in reference order, so the colour
  // classes (and hence MC chains) do not depend on the device site order
  for (int h = 0; h < N; ++h) {
    const int i = slot_of(c, h);
    for (int n : adj[i])
      if (col[n] >= 0) {
        if ((int)mark.size() <= col[n]) mark.resize(col[n] + 1, -1);
        mark[col[n]] = h;
      }
    int k = 0;
    while (k < (int)mark.size() && mark[k] == h) ++k;
    col[i] = k;
    ncol = std::max(ncol, k + 1);
  }
  for (int i = 0; i < N; ++i)
    for (int n : adj[i])
      if (col[n] == col[i]) return fail(UASD_ERR_ARG, "colouring failed (self-bond?)");
  c->ncolors = ncol;
  c->color_of_site = col;
  c->color_ptr.assign(ncol + 1, 0);
  for (int i = 0; i < N; ++i) c->color_ptr[col[i] + 1]++;
  for (int k = 0; k < ncol; ++k) c->color_ptr[k + 1] += c->color_ptr[k];
  c->color_sites.assign(N, 0);
  std::vector<int> fillp(c->color_ptr.begin(), c->color_ptr.end() - 1);
  for (int i = 0; i < N; ++i) c->color_sites[fillp[col[i]]++] = i;
  c->color_start.assign(ncol, 0);
  c->color_stride.assign(ncol, 0);
  for (int k = 0; k < ncol; ++k) {
    const int p0 = c->color_ptr[k], n = c->color_ptr[k + 1] - p0;
    if (n == 0) continue;
    const int a0 = c->color_sites[p0], d = n > 1 ? c->color_sites[p0 + 1] - a0 : 1;
    bool ap = d > 0;
    for (int i = 2; ap && i < n; ++i)
      ap = c->color_sites[p0 + i] - c->color_sites[p0 + i - 1] == d;
    c->color_start[k] = a0;
    c->color_stride[k] = ap ? d : 0;
  }
  c->coloring_dirty = false;
  c->col_version += 1;
  c->gen += 1;
  return UASD_OK;
}

}  // namespace

// Slot-major int16 entries of a slot-major list of device slots (see NbDec):
// v = delta * 2^kb + beta with beta = (b' - b) mod na and delta = (c' - c)
// mod nc taken in [-nc/2, nc/2).  False when any delta does not fit.
bool diff16(const uasd_ctx *c, const std::vector<int> &nb, int N, int W,
            std::vector<int16_t> &out) {
  const int na = c->order_na, nc = na == 1 ? N : c->order_nc, kb = idx_kb(c);
  const long lim = 1L << (15 - kb);
  out.resize((size_t)W * N);
  for (int j = 0; j < W; ++j)
    for (int d = 0; d < N; ++d) {
      const int n = nb[(size_t)j * N + d];
      const int b = d / nc, cc = d - b * nc, b2 = n / nc, c2 = n - b2 * nc;
      const int beta = ((b2 - b) % na + na) % na;
      long delta = (long)c2 - cc;
      if (2 * delta >= nc) delta -= nc;
      if (2 * delta < -(long)nc) delta += nc;
      if (delta < -lim || delta >= lim) return false;
      out[(size_t)j * N + d] = (int16_t)(delta * (1L << kb) + beta);
    }
  return true;
}

// ------------------------------------------------------------ stencil
// True when the list (device order) is one translation of a per-basis
// stencil over the periodic lattice; fills st.
bool detect_stencil(const uasd_ctx *c, const std::vector<int> &nb, const std::vector<int> &row,
                    const std::vector<int> &len, int W, uasd_ctx::Stencil &st) {
  const int NA = c->lat_na, N1 = c->lat_n1, N2 = c->lat_n2, N3 = c->lat_n3, N = c->N;
  st = uasd_ctx::Stencil{};
  if (NA <= 0 || W <= 0 || row.empty()) return false;
  st.W = W;
  st.bp.assign((size_t)NA * W, 0);
  st.dx = st.dy = st.dz = st.bp;
  auto wrap = [](int d, int n) { return 2 * d > n ? d - n : d; };
  std::vector<int> L(NA);
  for (int b = 0; b < NA; ++b) {
    const int d0 = slot_of(c, b);
    L[b] = len[row[d0]];
    for (int j = 0; j < L[b]; ++j) {
      const int n = site_of(c, nb[(size_t)j * N + d0]);
      const int bb = n % NA, cell = n / NA;
      const int x = cell % N1, y = (cell / N1) % N2, z = cell / (N1 * N2);
      st.bp[b * W + j] = bb;
      st.dx[b * W + j] = wrap(x, N1);
      st.dy[b * W + j] = wrap(y, N2);
      st.dz[b * W + j] = wrap(z, N3);
    }
  }
  for (int i = 0; i < N; ++i) {
    const int b = i % NA, cell = i / NA;
    const int x = cell % N1, y = (cell / N1) % N2, z = cell / (N1 * N2);
    const int d = slot_of(c, i);
    if (len[row[d]] != L[b]) return false;
    for (int j = 0; j < L[b]; ++j) {
      const int k = b * W + j;
      const int xx = ((x + st.dx[k]) % N1 + N1) % N1, yy = ((y + st.dy[k]) % N2 + N2) % N2,
                zz = ((z + st.dz[k]) % N3 + N3) % N3;
      const int want = st.bp[k] + NA * (xx + N1 * (yy + N2 * zz));
      if (site_of(c, nb[(size_t)j * N + d]) != want) return false;
    }
  }
  for (size_t k = 0; k < st.bp.size(); ++k) {
    st.rx = std::max(st.rx, std::abs(st.dx[k]));
    st.ry = std::max(st.ry, std::abs(st.dy[k]));
    st.rz = std::max(st.rz, std::abs(st.dz[k]));
  }
  st.ok = true;
  return true;
}

void build_stencil(uasd_ctx *c) {
  if (!c->stencil_dirty) return;
  c->stencil_dirty = false;
  c->stencil_ok = false;
  if (c->lat_na <= 0 || !c->have_ex) return;
  if (!detect_stencil(c, c->nbr_host, c->ex_row_of_site, c->ex_len_host, c->W, c->st_ex)) return;
  if (c->Wd > 0 && !detect_stencil(c, c->dnbr_host, c->dm_row_of_site, c->dm_len_host, c->Wd,
                                   c->st_dm))
    return;
  c->stencil_ok = true;
}

// Tile shape k (1-based) usable for this lattice and precision?
bool tile_fits(const uasd_ctx *c, int k) {
  if (!c->stencil_ok || k < 1 || k > uasd::kNumTileShapes) return false;
  // quad indices of the staging tables and the (tile, ensemble) units in int
  if ((int64_t)c->N * c->M >= (int64_t)1 << 31) return false;
  if (c->order_na != 1 && c->order_na != c->lat_na) return false;  // tile kernel's slot formula
  const int *sh = uasd::kTileShapes[k - 1];
  if ((c->lat_n3 > 1) != (sh[2] > 1)) return false;
  const int rx = std::max(c->st_ex.rx, c->st_dm.rx), ry = std::max(c->st_ex.ry, c->st_dm.ry),
            rz = std::max(c->st_ex.rz, c->st_dm.rz);
  const int hv = (sh[0] + 2 * rx) * (sh[1] + 2 * ry) * (sh[2] + 2 * rz);
  // one thread per site; whole wavefronts per basis atom
  if (sh[0] * sh[1] * sh[2] * c->lat_na > 1024 || (sh[0] * sh[1] * sh[2]) % 64 != 0) return false;
  const int plane = uasd::tile_plane(hv * c->lat_na);
  if (plane == 0) return false;
  // halo coordinates in FP32 reciprocal divisions: dividends below 2^22
  if (c->lat_n1 >= (1 << 20) || c->lat_n2 >= (1 << 20) || c->lat_n3 >= (1 << 20)) return false;
  // tile index arithmetic in FP32 reciprocals: fewer than 2^22 tiles
  if ((int64_t)((c->lat_n1 + sh[0] - 1) / sh[0]) * ((c->lat_n2 + sh[1] - 1) / sh[1]) *
          ((c->lat_n3 + sh[2] - 1) / sh[2]) >= (1 << 22))
    return false;
  const int ntab = sh[0] + 2 * rx + c->lat_na * (sh[1] + 2 * ry) * (sh[2] + 2 * rz);
  if ((sh[0] + 2 * rx) > sh[0] * sh[1] * sh[2] * c->lat_na) return false;  // a row per round
  return (int64_t)uasd::tile_lds_bytes(c->rsize, plane, ntab) <= c->lds_max;
}

// TileDev for shape k, uploading its halo offsets when the shape changes.
int make_tile(uasd_ctx *c, int k, uasd::TileDev &t) {
  const int *sh = uasd::kTileShapes[k - 1];
  t = uasd::TileDev{};
  t.N1 = c->lat_n1;
  t.N2 = c->lat_n2;
  t.N3 = c->lat_n3;
  t.NA = c->lat_na;
  t.TX = sh[0];
  t.TY = sh[1];
  t.TZ = sh[2];
  t.RX = std::max(c->st_ex.rx, c->st_dm.rx);
  t.RY = std::max(c->st_ex.ry, c->st_dm.ry);
  t.RZ = std::max(c->st_ex.rz, c->st_dm.rz);
  t.HX = t.TX + 2 * t.RX;
  t.HY = t.TY + 2 * t.RY;
  t.HZ = t.TZ + 2 * t.RZ;
  t.HV = t.HX * t.HY * t.HZ;
  t.rTX = 1.0f / (float)t.TX;
  t.rTXY = 1.0f / (float)(t.TX * t.TY);
  t.rTC = 1.0f / (float)(t.TX * t.TY * t.TZ);
  t.rHX = 1.0f / (float)t.HX;
  t.rs = t.TX * t.TY * t.TZ * t.NA / t.HX;  // halo rows staged per round
  t.ntx = (t.N1 + t.TX - 1) / t.TX;
  t.nty = (t.N2 + t.TY - 1) / t.TY;
  t.ntz = (t.N3 + t.TZ - 1) / t.TZ;
  t.rntx = 1.0f / (float)t.ntx;
  t.rntxy = 1.0f / (float)(t.ntx * t.nty);
  t.rHY = 1.0f / (float)t.HY;
  t.rHYZ = 1.0f / (float)(t.HY * t.HZ);
  t.rN1 = 1.0f / (float)t.N1;
  t.rN2 = 1.0f / (float)t.N2;
  t.rN3 = 1.0f / (float)t.N3;
  t.ox = t.N1 * ((t.RX + t.N1 - 1) / t.N1);
  t.oy = t.N2 * ((t.RY + t.N2 - 1) / t.N2);
  t.oz = t.N3 * ((t.RZ + t.N3 - 1) / t.N3);
  t.W = c->st_ex.W;
  t.Wd = c->Wd > 0 ? c->st_dm.W : 0;
  if (c->tile_off_shape != k) {
    std::vector<int> off((size_t)t.NA * (t.W + t.Wd), 0);
    auto fill = [&](const uasd_ctx::Stencil &st, int W, int base) {
      for (int b = 0; b < t.NA; ++b)
        for (int j = 0; j < W; ++j) {
          const int q = b * W + j;
          off[base + q] = st.bp[q] * t.HV + st.dz[q] * t.HX * t.HY + st.dy[q] * t.HX + st.dx[q];
        }
    };
    fill(c->st_ex, t.W, 0);
    if (t.Wd > 0) fill(c->st_dm, t.Wd, t.NA * t.W);
    if (int r = upload_raw(c, c->tile_off, off)) return r;
    c->tile_off_shape = k;
  }
  t.off = c->tile_off.as<int>();
  t.doff = t.off + (size_t)t.NA * t.W;
  // one site class per basis atom? (checked once per class rebuild)
  if (c->ucls_version != c->cls_version) {
    c->ucls = 0;
    if (t.NA <= 8 && (int)c->cls_host.size() == c->N) {
      c->ucls = 1;
      for (int b = 0; b < t.NA; ++b) c->cls_b[b] = c->cls_host[slot_of(c, b)];
      for (int i = 0; i < c->N && c->ucls; ++i)
        if (c->cls_host[slot_of(c, i)] != c->cls_b[i % t.NA]) c->ucls = 0;
    }
    c->ucls_version = c->cls_version;
  }
  t.ucls = c->ucls;
  for (int b = 0; b < 8; ++b) t.cls_b[b] = c->cls_b[b];
  return UASD_OK;
}

// ------------------------------------------------------------ segments
// Sites per reduction chunk, one workgroup each: the fewest, from 256 (a site
// per thread) up to 4096, whose partial sums fit the fixed scratch of
// uasd_energy_terms_noalloc, so that entry point sums in the same order as
// uasd_energy_terms.  Small chunks fill the chip: calc_energy's terms of
// 221,184 sites with 58 neighbours took 202 us in 54 chunks of 4096 sites (54
// workgroups cannot fill 256 CUs) and take 45 us in 864 chunks of 256.
constexpr int kSegChunkMax = 4096;

int seg_chunk_size(int nseg, const int *off, int M) {
  int size = 256;
  for (; size < kSegChunkMax; size *= 2) {
    size_t n = nseg;
    for (int s = 0; s < nseg; ++s) n += ((size_t)(off[s + 1] - off[s]) + size - 1) / size;
    if (n * M * 4 <= kScratchDoubles) break;
  }
  return size;
}

int set_segments(uasd_ctx *c, int nseg, const int *off) {
  std::vector<int> chunks, seg_chunk(1, 0), seg_n;
  const int size = seg_chunk_size(nseg, off, c->M);
  for (int s = 0; s < nseg; ++s) {
    for (int a = off[s]; a < off[s + 1]; a += size) {
      chunks.push_back(a);
      chunks.push_back(std::min(off[s + 1], a + size));
    }
    seg_chunk.push_back((int)chunks.size() / 2);
    seg_n.push_back(off[s + 1] - off[s]);
  }
  std::vector<int> all(chunks);
  all.insert(all.end(), seg_chunk.begin(), seg_chunk.end());
  all.insert(all.end(), seg_n.begin(), seg_n.end());
  if (int r = upload_raw(c, c->seg_dev, all)) return r;
  c->nseg = nseg;
  c->seg_off.assign(off, off + nseg + 1);
  c->nchunks = (int)chunks.size() / 2;
  const size_t nacc = (size_t)nseg * c->M * uasd::kAccWidth;
  HIP_TRY(c->acc.ensure(nacc * sizeof(double)));
  std::vector<double> zero(nacc, 0.0);  // uploaded, not memset: the accumulators
  if (int r = upload_raw(c, c->acc, zero)) return r;  // may later sit under a graph
  c->acc_samples = 0;
  return UASD_OK;
}

int ensure_segments(uasd_ctx *c) {
  if (c->nseg > 0) return UASD_OK;
  const int off[2] = {0, c->N};
  return set_segments(c, 1, off);
}

// Per-(segment, ensemble) FP64 sums into c->seg_out; energy terms from the
// last field launch when with_energy.  Asynchronous.
template <typename R>
int segment_sums(uasd_ctx *c, bool with_energy) {
  const int nv = with_energy ? 4 : 3;
  HIP_TRY(c->seg_partial.ensure((size_t)c->nchunks * c->M * nv * sizeof(double)));
  HIP_TRY(c->seg_out.ensure((size_t)c->nseg * c->M * 4 * sizeof(double)));
  const int2 *chunks = c->seg_dev.as<int2>();
  const int *seg_chunk = reinterpret_cast<const int *>(chunks + c->nchunks);
  HIP_TRY(uasd::launch_segsum<R>(c->stream, c->M, c->nseg, c->nchunks, chunks, seg_chunk,
                                 quads<R>(c, c->spins, 0),
                                 with_energy ? c->energy.as<double>() : nullptr, nv,
                                 c->seg_partial.as<double>(), c->seg_out.as<double>()));
  return UASD_OK;
}

// =================================================================== C-ABI
extern "C" {

const char *uasd_last_error(void) { return g_err.c_str(); }

int uasd_version(void) { return UASD_API_VERSION; }

int uasd_device_count(int *count) {
  if (!count) return fail(UASD_ERR_ARG, "count is null");
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) n = 0;
  *count = n;
  return UASD_OK;
}

int uasd_ctx_create(uasd_ctx **out, int natom, int mensemble, int precision) {
  if (!out) return fail(UASD_ERR_ARG, "out is null");
  *out = nullptr;
  if (natom <= 0 || mensemble <= 0) return fail(UASD_ERR_ARG, "natom and mensemble must be > 0");
  if ((int64_t)natom * mensemble > (int64_t)1 << 31)
    return fail(UASD_ERR_ARG, "natom*mensemble exceeds 2^31");
  if (precision != UASD_FP64 && precision != UASD_FP32)
    return fail(UASD_ERR_ARG, "precision must be UASD_FP64 or UASD_FP32");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return fail(UASD_ERR_NODEVICE, "no HIP device available");
  auto c = std::make_unique<uasd_ctx>();
  c->N = natom;
  c->M = mensemble;
  c->prec = precision;
  c->rsize = precision == UASD_FP64 ? 8 : 4;
  HIP_TRY(hipGetDevice(&c->device));
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, c->device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(UASD_ERR_NODEVICE, std::string("device is ") + prop.gcnArchName +
                                       ", the library is built for gfx950");
  c->lds_max = (int64_t)std::max(prop.sharedMemPerBlock, prop.sharedMemPerBlockOptin);
  if (int r = scratch_init(c->device)) return r;
  HIP_TRY(hipStreamCreateWithFlags(&c->own_stream, hipStreamNonBlocking));
  c->stream = c->own_stream;
  HIP_TRY(c->spins.ensure(2 * quad_bytes(c.get()) + raw_room(c.get())));
  HIP_TRY(hipMemsetAsync(c->spins.p, 0, 3 * quad_bytes(c.get()), c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  // (here, not with the first replay, which may come unasked for: another
  // thread's capture can forbid allocations)
  HIP_TRY(c->ctr.ensure(2 * sizeof(uint64_t)));
  // the whole lattice as one segment until uasd_set_segments says otherwise
  if (int r = ensure_segments(c.get())) return r;
  *out = c.release();
  return UASD_OK;
}

int uasd_ctx_destroy(uasd_ctx *c) {
  if (!c) return UASD_OK;
  // the context is released whatever happens; a failure of the work still
  // queued on its stream is reported, the release calls' own are not
  const hipError_t serr = c->stream ? hipStreamSynchronize(c->stream) : hipSuccess;
  for (const auto &pe : c->pending) {  // timings not yet read are dropped
    (void)hipEventDestroy(pe.a);
    (void)hipEventDestroy(pe.b);
  }
  destroy_graphs(c);
  if (c->cur) (void)hipEventDestroy(c->cur);
  if (c->region_cur) (void)hipEventDestroy(c->region_cur);
  for (hipEvent_t e : c->ev_pool) (void)hipEventDestroy(e);
  if (c->own_stream) (void)hipStreamDestroy(c->own_stream);
  delete c;
  if (serr != hipSuccess)
    return fail(UASD_ERR_HIP, std::string("uasd_ctx_destroy: queued work failed: ") +
                                  hipGetErrorString(serr));
  return UASD_OK;
}

int uasd_ctx_set_stream(uasd_ctx *c, void *s) {
  if (int r = check_ctx(c)) return r;
  HIP_TRY(hipStreamSynchronize(c->stream));
  c->stream = s ? static_cast<hipStream_t>(s) : c->own_stream;
  c->replays_off = false;
  return UASD_OK;
}

void *uasd_ctx_stream(uasd_ctx *c) { return c ? (void *)c->stream : nullptr; }

int uasd_ctx_sync(uasd_ctx *c) {
  if (int r = check_ctx(c)) return r;
  HIP_TRY(hipStreamSynchronize(c->stream));
  return UASD_OK;
}

int uasd_set_exchange(uasd_ctx *c, int mnn, int nham, const int *nlist, const int *nlistsize,
                      const double *ncoup, const int *aham) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  const int N = c->N;
  if (mnn < 0 || nham <= 0 || !nlist || !nlistsize || (mnn > 0 && !ncoup))
    return fail(UASD_ERR_ARG, "uasd_set_exchange: bad arguments");
  std::vector<int> ref(N);
  for (int i = 0; i < N; ++i) {
    int r = aham ? aham[i] - 1 : i;
    if (r < 0 || r >= nham) return fail(UASD_ERR_ARG, "aham entry out of range");
    if (nlistsize[r] < 0 || nlistsize[r] > mnn) return fail(UASD_ERR_ARG, "nlistsize > max_no_neigh");
    ref[i] = r;
  }
  RowSet rs = dedupe_rows(N, ref, nlistsize, ncoup, mnn, 1);
  int W = 0;
  for (int L : rs.len) W = std::max(W, L);
  // device order: slot d = slot_of(i) holds site i; list values are slots
  std::vector<int> nb((size_t)std::max(W, 1) * N), row_dev(N);
  for (int i = 0; i < N; ++i) {
    const int d = slot_of(c, i);
    int L = rs.len[rs.row_of_site[i]];
    row_dev[d] = rs.row_of_site[i];
    for (int j = 0; j < W; ++j) {
      int v = d;
      if (j < L) {
        v = nlist[(size_t)j + (size_t)mnn * i] - 1;
        if (v < 0 || v >= N) return fail(UASD_ERR_ARG, "nlist entry out of range");
        v = slot_of(c, v);
      }
      nb[(size_t)j * N + d] = v;
    }
  }
  const int rows = (int)rs.len.size();
  std::vector<double> cp((size_t)std::max(W, 1) * rows, 0.0);
  for (int r = 0; r < rows; ++r)
    for (int j = 0; j < rs.len[r]; ++j) cp[(size_t)j * rows + r] = rs.vals[r][j];
  c->W = W;
  c->ex_rows = rows;
  c->ex_row_of_site = row_dev;
  c->ex_len_host = rs.len;
  c->ex_full = W > 0 && std::all_of(rs.len.begin(), rs.len.end(), [W](int l) { return l == W; });
  c->nbr_host = nb;
  if (int r = upload_raw(c, c->nbr, nb)) return r;
  std::vector<int16_t> d16;
  c->use16 = W > 0 && diff16(c, nb, N, W, d16);
  if (c->use16) {
    if (int r = upload_raw(c, c->nbr16, d16)) return r;
  } else {
    c->nbr16.release();
  }
  if (int r = upload_raw(c, c->ex_len, rs.len)) return r;
  if (int r = upload_real(c, c->cpl, cp)) return r;
  c->have_ex = true;
  c->classes_dirty = true;
  c->coloring_dirty = true;
  c->stencil_dirty = true;
  c->tile_off_shape = 0;
  return UASD_OK;
}

int uasd_set_dm(uasd_ctx *c, int mdm, int nham, const int *dmlist, const int *dmlistsize,
                const double *dm_vect, const int *aham) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  const int N = c->N;
  if (!dmlist || mdm <= 0) {  // clear
    c->Wd = 0;
    c->dm_rows = 0;
    c->dm_row_of_site.clear();
    c->classes_dirty = c->coloring_dirty = true;
  c->stencil_dirty = true;
  c->tile_off_shape = 0;
    return UASD_OK;
  }
  if (nham <= 0 || !dmlistsize || !dm_vect) return fail(UASD_ERR_ARG, "uasd_set_dm: bad arguments");
  std::vector<int> ref(N);
  for (int i = 0; i < N; ++i) {
    int r = aham ? aham[i] - 1 : i;
    if (r < 0 || r >= nham) return fail(UASD_ERR_ARG, "aham entry out of range");
    if (dmlistsize[r] < 0 || dmlistsize[r] > mdm) return fail(UASD_ERR_ARG, "dmlistsize > max");
    ref[i] = r;
  }
  RowSet rs = dedupe_rows(N, ref, dmlistsize, dm_vect, mdm, 3);
  int W = 0;
  for (int L : rs.len) W = std::max(W, L);
  std::vector<int> nb((size_t)std::max(W, 1) * N), row_dev(N);
  for (int i = 0; i < N; ++i) {
    const int d = slot_of(c, i);
    int L = rs.len[rs.row_of_site[i]];
    row_dev[d] = rs.row_of_site[i];
    for (int j = 0; j < W; ++j) {
      int v = d;
      if (j < L) {
        v = dmlist[(size_t)j + (size_t)mdm * i] - 1;
        if (v < 0 || v >= N) return fail(UASD_ERR_ARG, "dmlist entry out of range");
        v = slot_of(c, v);
      }
      nb[(size_t)j * N + d] = v;
    }
  }
  const int rows = (int)rs.len.size();
  const size_t n = (size_t)std::max(W, 1) * rows;
  std::vector<double> dv(3 * n, 0.0);
  for (int r = 0; r < rows; ++r)
    for (int j = 0; j < rs.len[r]; ++j)
      for (int d = 0; d < 3; ++d) dv[d * n + (size_t)j * rows + r] = rs.vals[r][3 * j + d];
  c->Wd = W;
  c->dm_rows = rows;
  c->dm_row_of_site = row_dev;
  c->dm_len_host = rs.len;
  c->dnbr_host = nb;
  if (int r = upload_raw(c, c->dnbr, nb)) return r;
  std::vector<int16_t> d16;
  c->use16_dm = W > 0 && diff16(c, nb, N, W, d16);
  if (c->use16_dm) {
    if (int r = upload_raw(c, c->dnbr16, d16)) return r;
  } else {
    c->dnbr16.release();
  }
  if (int r = upload_raw(c, c->dm_len, rs.len)) return r;
  if (int r = upload_real(c, c->dv, dv)) return r;
  c->classes_dirty = c->coloring_dirty = true;
  c->stencil_dirty = true;
  c->tile_off_shape = 0;
  return UASD_OK;
}

int uasd_set_anisotropy(uasd_ctx *c, const int *taniso, const double *eaniso,
                        const double *kaniso, const double *sb) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  const int N = c->N;
  if (!taniso) {
    c->an_rows = 0;
    c->an_row_of_site.clear();
    c->classes_dirty = true;
    return UASD_OK;
  }
  if (!eaniso || !kaniso || !sb) return fail(UASD_ERR_ARG, "uasd_set_anisotropy: null array");
  std::map<std::vector<double>, int> rows;
  std::vector<int> row_of(N, -1);
  std::vector<std::vector<double>> vals;
  std::vector<int> types;
  for (int i = 0; i < N; ++i) {
    int t = taniso[i];
    if (t != 0 && t != 1 && t != 2 && t != 7)
      return fail(UASD_ERR_UNSUPPORTED, "anisotropy type must be 0, 1, 2 or 7");
    if (t == 0) continue;
    std::vector<double> key = {(double)t,     eaniso[3 * (size_t)i], eaniso[3 * (size_t)i + 1],
                               eaniso[3 * (size_t)i + 2], kaniso[2 * (size_t)i],
                               kaniso[2 * (size_t)i + 1], sb[i]};
    auto it = rows.find(key);
    if (it == rows.end()) {
      it = rows.emplace(key, (int)vals.size()).first;
      vals.push_back(key);
      types.push_back(t);
    }
    row_of[i] = it->second;
  }
  const int nr = (int)vals.size();
  c->an_rows = nr;
  c->an_row_of_site.assign(N, -1);
  for (int i = 0; i < N; ++i) c->an_row_of_site[slot_of(c, i)] = row_of[i];
  if (nr > 0) {
    std::vector<double> v(6 * (size_t)nr);
    for (int r = 0; r < nr; ++r)
      for (int k = 0; k < 6; ++k) v[(size_t)k * nr + r] = vals[r][1 + k];
    if (int r = upload_raw(c, c->an_type, types)) return r;
    if (int r = upload_real(c, c->an_vals, v)) return r;
  }
  c->classes_dirty = true;
  return UASD_OK;
}

int uasd_set_external_field(uasd_ctx *c, const double *field) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  const int N = c->N, M = c->M;
  if (!field) {
    c->ext_mode = 0;
    c->ext_u_host.assign(3 * (size_t)M, 0.0);
    return upload_real(c, c->ext_u, c->ext_u_host);
  }
  bool uniform = true, zero = true;
  for (int k = 0; k < M && uniform; ++k) {
    const double *f0 = field + 3 * ((size_t)N * k);
    for (int i = 0; i < N && uniform; ++i) {
      const double *f = field + 3 * ((size_t)i + (size_t)N * k);
      for (int d = 0; d < 3; ++d) {
        if (std::memcmp(&f[d], &f0[d], sizeof(double)) != 0) uniform = false;
        if (f[d] != 0.0) zero = false;
      }
    }
  }
  c->ext_u_host.assign(3 * (size_t)M, 0.0);
  if (uniform) {
    for (int k = 0; k < M; ++k)
      for (int d = 0; d < 3; ++d) c->ext_u_host[3 * k + d] = field[3 * ((size_t)N * k) + d];
    c->ext_mode = zero ? 0 : 1;
    return upload_real(c, c->ext_u, c->ext_u_host);
  }
  c->ext_mode = 2;
  if (int r = upload_real(c, c->ext_u, c->ext_u_host)) return r;
  HostIo io(c);
  if (int r = upload_vec(io, c->ext_full, 0, field, PackW{})) return r;
  return io.wait();
}

int uasd_set_llg(uasd_ctx *c, const double *lambda1, const double *temp, const double *landeg,
                 double delta_t, double temprescale, double bn) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  const int N = c->N;
  if (!lambda1 || !temp) return fail(UASD_ERR_ARG, "uasd_set_llg: lambda1 and temp required");
  if (!(delta_t > 0.0)) return fail(UASD_ERR_ARG, "delta_t must be > 0");
  auto is_uniform = [N](const double *a) {
    for (int i = 1; i < N; ++i)
      if (std::memcmp(&a[i], &a[0], sizeof(double)) != 0) return false;
    return true;
  };
  std::vector<double> arr(3 * (size_t)N);
  for (int i = 0; i < N; ++i) {
    const int d = slot_of(c, i);
    arr[d] = lambda1[i];
    arr[N + d] = temp[i];
    arr[2 * (size_t)N + d] = landeg ? landeg[i] : 1.0;
  }
  c->lam_uniform = is_uniform(lambda1);
  c->temp_uniform = is_uniform(temp);
  c->lande_uniform = landeg ? is_uniform(landeg) : true;
  c->lam0 = lambda1[0];
  c->temp0 = temp[0];
  c->lande0 = landeg ? landeg[0] : 1.0;
  c->dt = delta_t;
  c->temprescale = temprescale;
  c->bn = bn;
  if (int r = upload_raw(c, c->llgarr, arr)) return r;
  c->have_llg = true;
  return UASD_OK;
}

int uasd_set_temprescale(uasd_ctx *c, double temprescale) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  if (!(temprescale > 0.0)) return fail(UASD_ERR_ARG, "temprescale must be > 0");
  c->temprescale = temprescale;
  return UASD_OK;
}

int uasd_set_noise(uasd_ctx *c, int mode, uint64_t seed, const double *normals) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  if (mode != UASD_NOISE_NONE && mode != UASD_NOISE_PHILOX && mode != UASD_NOISE_INJECTED)
    return fail(UASD_ERR_ARG, "unknown noise mode");
  if (mode == UASD_NOISE_INJECTED) {
    if (!normals) return fail(UASD_ERR_ARG, "injected noise needs the normals array");
    HostIo io(c);
    if (int r = upload_vec(io, c->noise, 0, normals, PackW{})) return r;
    if (int r = io.wait()) return r;
  }
  if (mode == UASD_NOISE_PHILOX && (seed != c->seed || c->noise_mode != mode)) c->step = 0;
  c->noise_mode = mode;
  c->seed = seed;
  return UASD_OK;
}

int uasd_set_moments(uasd_ctx *c, const double *emom, const double *mmom) {
  if (int r = check_ctx(c)) return r;
  if (!emom || !mmom) return fail(UASD_ERR_ARG, "uasd_set_moments: null array");
  HostIo io(c);
  io.open = true;
  // the raw arrays (32 bytes a pair) pass through the memory of b2eff, which
  // lasts no longer than a step: a call that every program makes once needs no
  // staging of its own
  const size_t pairs = (size_t)c->N * c->M, step = raw_room(c) / kRawMoment;
  double *sa = reinterpret_cast<double *>(static_cast<char *>(c->spins.p) + 2 * quad_bytes(c));
  for (size_t p0 = 0; p0 < pairs; p0 += step) {
    const size_t n = std::min(step, pairs - p0);
    HIP_TRY(hipMemcpyAsync(sa, emom + 3 * p0, 3 * n * sizeof(double), hipMemcpyHostToDevice,
                           c->stream));
    HIP_TRY(hipMemcpyAsync(sa + 3 * n, mmom + p0, n * sizeof(double), hipMemcpyHostToDevice,
                           c->stream));
    // emom2 starts as emom
    if (int r = launch_pack(c, c->spins, 0, p0, n, sa, sa + 3 * n, PackW{}, true)) return r;
  }
  if (int r = io.wait()) return r;
  c->have_state = true;
  const size_t nm = (size_t)c->N * c->M;
  c->m_uniform = std::all_of(mmom, mmom + nm, [&](double v) { return v == mmom[0]; });
  c->m0 = mmom[0];
  c->gen += 1;  // captured steps hold the noise amplitudes
  return UASD_OK;
}

int uasd_get_moments(uasd_ctx *c, double *emom, double *emomM) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_state) return fail(UASD_ERR_STATE, "moments not set");
  HostIo io(c);
  if (emom)
    if (int r = download_vec(io, c->spins, 0, emom, false)) return r;
  if (emomM)
    if (int r = download_vec(io, c->spins, 0, emomM, true)) return r;
  return io.wait();
}

// ---------------------------------------------------------- drop-in (host)
// Host vec3 arrays are uploaded as quads; spin quads keep the resident mmom
// in w, the others carry a constant.

// quad array k of the spins <- the (3,N,M) array a, with w = mmom of the
// state (quad array 0): the magnitudes stay on the device
static int upload_vec_keep_w(HostIo &io, int k, const double *a) {
  return upload_vec(io, io.c->spins, k, a, PackW{1, 0.0});
}

int uasd_effective_field_host(uasd_ctx *c, const double *emomM, double *beff, double *beff1,
                              double *beff2, double *energy) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_ex) return fail(UASD_ERR_STATE, "exchange not set");
  if (!emomM || !beff) return fail(UASD_ERR_ARG, "null array");
  if (int r = rebuild_classes(c)) return r;
  HostIo io(c);
  if (int r = upload_vec(io, c->scratch, 0, emomM, PackW{0, 1.0})) return r;
  const bool parts = beff1 || beff2;
  int r = c->prec == UASD_FP64 ? run_field<double>(c, true, energy != nullptr, parts)
                               : run_field<float>(c, true, energy != nullptr, parts);
  if (r) return r;
  if ((r = download_vec(io, c->field, 0, beff, false))) return r;
  if (beff1 && (r = download_vec(io, c->field, 1, beff1, false))) return r;
  if (beff2 && (r = download_vec(io, c->field, 2, beff2, false))) return r;
  if (energy) {
    std::vector<double> red;
    r = c->prec == UASD_FP64 ? reduce_moments<double>(c, true, true, red)
                             : reduce_moments<float>(c, true, true, red);
    if (r) return r;
    double e = 0.0;
    for (int k = 0; k < c->M; ++k) e += red[4 * (size_t)k + 3];
    *energy = e * uasd::kMub / uasd::kMry;
  }
  return io.wait();
}

int uasd_evolve_first_host(uasd_ctx *c, int alg, const double *beff, double *emom, double *emom2,
                           double *emomM, double *b2eff) {
  if (int r = check_ctx(c)) return r;
  if (!sde_supported(alg))
    return fail(UASD_ERR_UNSUPPORTED, "SDEalgh must be 1 (midpoint), 4 (Heun), 5 (Depondt), 6 (SIB) or 7 (spherical midpoint)");
  if (!beff || !emom || !emom2 || !emomM || (sde_b2eff(alg) && !b2eff))
    return fail(UASD_ERR_ARG, "null array");
  if (int r = ready_for_llg(c)) return r;
  HostIo io(c);
  if (int r = upload_vec(io, c->field, 0, beff, PackW{})) return r;
  // heun4p starts from emom2 (heun_proper.f90:309-311), the others from emom
  if (int r = upload_vec_keep_w(io, 0, alg == UASD_SDE_HEUN ? emom2 : emom)) return r;
  int r = c->prec == UASD_FP64 ? run_llg_half<double>(c, alg, 0, false, false)
                               : run_llg_half<float>(c, alg, 0, false, false);
  if (r) return r;
  if (alg == UASD_SDE_DEPONDT) {
    // depondt.f90:182-187: emom2 = m(t), emom = rotated, emomM = emom*mmom, b2eff = bdup
    if ((r = io.wait())) return r;  // emom has been read before it is written
    std::memcpy(emom2, emom, sizeof(double) * 3 * (size_t)c->N * c->M);
    if ((r = download_vec(io, c->spins, 1, emom, false))) return r;
    if ((r = download_vec(io, c->spins, 2, b2eff, false))) return r;
  } else if (alg == UASD_SDE_HEUN) {
    // heun_proper.f90:303-365: b2eff = beff, emom = predictor, emomM =
    // emom*mmom, emom2 unchanged
    if ((r = download_vec(io, c->spins, 1, emom, false))) return r;
    if ((r = download_vec(io, c->spins, 2, b2eff, false))) return r;
  } else {
    // midpoint.f90:167-175 (and sibt / sispht, sphmidpoint.f90:247-258,
    // 698-710): emom2 = et', emomM = et'*mmom, emom unchanged
    if ((r = download_vec(io, c->spins, 1, emom2, false))) return r;
  }
  if ((r = download_vec(io, c->spins, 1, emomM, true))) return r;
  return io.wait();
}

int uasd_evolve_second_host(uasd_ctx *c, int alg, const double *beff, const double *b2eff,
                            double *emom, double *emom2) {
  if (int r = check_ctx(c)) return r;
  if (!sde_supported(alg))
    return fail(UASD_ERR_UNSUPPORTED, "SDEalgh must be 1 (midpoint), 4 (Heun), 5 (Depondt), 6 (SIB) or 7 (spherical midpoint)");
  if (!beff || !emom || !emom2 || (sde_b2eff(alg) && !b2eff))
    return fail(UASD_ERR_ARG, "null array");
  if (int r = ready_for_llg(c)) return r;
  HostIo io(c);
  if (int r = upload_vec(io, c->field, 0, beff, PackW{})) return r;
  if (alg == UASD_SDE_DEPONDT || alg == UASD_SDE_HEUN) {
    // reference on entry: emom = predicted, emom2 = m(t)
    if (int r = upload_vec_keep_w(io, 1, emom)) return r;
    if (int r = upload_vec_keep_w(io, 0, emom2)) return r;
    if (int r = upload_vec(io, c->spins, 2, b2eff, PackW{})) return r;
  } else {
    if (int r = upload_vec_keep_w(io, 0, emom)) return r;
    if (int r = upload_vec_keep_w(io, 1, emom2)) return r;
  }
  int r = c->prec == UASD_FP64 ? run_llg_half<double>(c, alg, 1, false, false)
                               : run_llg_half<float>(c, alg, 1, false, false);
  if (r) return r;
  if (alg == UASD_SDE_DEPONDT) {
    if ((r = io.wait())) return r;  // both have been read before they are written
    std::memcpy(emom, emom2, sizeof(double) * 3 * (size_t)c->N * c->M);
  }
  if ((r = download_vec(io, c->spins, 1, emom2, false))) return r;
  if ((r = io.wait())) return r;
  c->step += 1;
  return UASD_OK;
}

// ----------------------------------------------------------- resident path
}  // extern "C"

namespace {

void destroy_graphs(uasd_ctx *c) {
  for (auto &kv : c->graphs) {
    if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
    if (kv.second.g) (void)hipGraphDestroy(kv.second.g);
  }
  c->graphs.clear();
}

// Whether the context stream is known not to be capturing.
bool stream_free(uasd_ctx *c) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(c->stream, &st) == hipSuccess) return st == hipStreamCaptureStatusNone;
  (void)hipGetLastError();  // not known: the next launch's error is its own
  return false;
}

// Builds the graph of what body() enqueues and instantiates it.  Not for a
// stream that a caller captures: its replays would not move the host's counter.
template <typename F>
int record_graph(uasd_ctx *c, F &&body, uasd_ctx::Graph &out) {
  if (!stream_free(c))
    return fail(UASD_ERR_HIP, "graphs of steps or sweeps need a stream that is not being captured");
  uasd::Recording rec;
  HIP_TRY(hipGraphCreate(&rec.graph, 0));
  c->rec = &rec;
  const int r = body();
  c->rec = nullptr;
  hipGraphExec_t x = nullptr;
  const hipError_t e = r ? hipSuccess : hipGraphInstantiate(&x, rec.graph, nullptr, nullptr, 0);
  if (r || e != hipSuccess) {
    (void)hipGraphDestroy(rec.graph);
    return r ? r : fail(UASD_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
  }
  out.g = rec.graph;
  out.exec = x;
  return UASD_OK;
}

// Replays graph `key` (built on first use), which advances device
// counter idx by K.  The device counter is first set to host_ctr when they
// differ (after eager steps), with a kernel, so no memset or copy node is
// ever recorded.
template <typename F>
int replay_graph(uasd_ctx *c, const std::tuple<int, int, int, uint64_t> &key, int idx,
                 uint64_t &host_ctr, int K, int timer, F &&body) {
  if (c->graphs_gen != c->gen || c->graphs.size() > 16) {
    // HIP does not say that a graph outlives its last handle while it runs:
    // the replays of an earlier call, which did not wait for them, end first
    if (!c->graphs.empty()) HIP_TRY(hipStreamSynchronize(c->stream));
    destroy_graphs(c);
    c->graphs_gen = c->gen;
  }
  auto it = c->graphs.find(key);
  if (it == c->graphs.end()) {
    uasd_ctx::Graph gr;
    if (int r = record_graph(c, body, gr)) return r;
    it = c->graphs.emplace(key, gr).first;
  }
  if (!c->ctr_valid[idx] || c->ctr_val[idx] != host_ctr) {
    HIP_TRY(uasd::launch_counter(queue(c), idx, c->ctr.as<uint64_t>(), host_ctr, 0));
    c->ctr_valid[idx] = true;
  }
  tic(c, timer);
  HIP_TRY(hipGraphLaunch(it->second.exec, c->stream));
  count(c, idx == 0 ? UASD_LAUNCH_LLG_GRAPH : UASD_LAUNCH_MC_GRAPH);
  if (int r = toc(c, timer)) return r;
  host_ctr += (uint64_t)K;
  c->ctr_val[idx] = host_ctr;
  return UASD_OK;
}

}  // namespace

extern "C" {

int uasd_set_graph_steps(uasd_ctx *c, int steps_per_graph) {
  if (int r = check_ctx(c)) return r;
  if (steps_per_graph < 0 || steps_per_graph > 4096)
    return fail(UASD_ERR_ARG, "steps_per_graph must be 0 (off) .. 4096");
  c->graph_steps = steps_per_graph;
  return UASD_OK;
}

int uasd_sd_steps(uasd_ctx *c, int alg, int64_t nsteps) {
  if (int r = check_ctx(c)) return r;
  if (!sde_supported(alg))
    return fail(UASD_ERR_UNSUPPORTED, "SDEalgh must be 1 (midpoint), 4 (Heun), 5 (Depondt), 6 (SIB) or 7 (spherical midpoint)");
  if (nsteps < 0) return fail(UASD_ERR_ARG, "nsteps < 0");
  if (int r = ready_for_llg(c)) return r;
  if (int r = region_tic(c)) return r;
  if (int r = sd_steps_run(c, alg, nsteps)) return r;
  return region_toc(c);
}

}  // extern "C"

namespace {

// An automatic replay that failed: nothing of it ran, so the call goes on with
// single launches, and no other replay is tried on this stream.
void replay_failed(uasd_ctx *c) {
  (void)hipGetLastError();
  c->replays_off = true;
}

// One LLG step, both halves; step_off, ahead as in run_llg_half.
int llg_step(uasd_ctx *c, int alg, int64_t step_off, int ahead) {
  const bool d = c->prec == UASD_FP64;
  for (int half = 0; half < 2; ++half) {
    const int r = d ? run_llg_half<double>(c, alg, half, true, half == 1, step_off, ahead)
                    : run_llg_half<float>(c, alg, half, true, half == 1, step_off, ahead);
    if (r) return r;
  }
  return UASD_OK;
}

// The tile shape the launched half steps take, 0 for the list kernels.
int launched_tile(uasd_ctx *c) {
  if (c->tune[0].tile == 0) return 0;
  build_stencil(c);
  return tile_fits(c, c->tune[0].tile) ? c->tune[0].tile : 0;
}

// Deviates of n steps (from the context's step, or inside a graph from
// *ctr[0] + step_off) into c->nsave.
template <typename R>
int draw_ahead(uasd_ctx *c, int n, int64_t step_off) {
  uasd::LLGDev<R> prm = llg_view<R>(c);
  if (step_off >= 0) {
    prm.step = (uint64_t)step_off;
    prm.step_dev = c->ctr.as<uint64_t>();
  }
  HIP_TRY(uasd::launch_draw<R>(queue(c), ham_view<R>(c), prm, n, quads<R>(c, c->nsave)));
  count(c, UASD_LAUNCH_DRAW);
  return UASD_OK;
}

// n LLG steps launched one by one; in_graph: inside a graph, counted from
// the device counter.
int llg_steps(uasd_ctx *c, int alg, int64_t n, bool in_graph) {
  int K = llg_view<double>(c).noise_mode == UASD_NOISE_PHILOX ? steps_ahead(c) : 1;
  if (launched_tile(c)) K = 1;  // the tile kernels draw their own deviates
  for (int64_t s = 0; s < n; ++s) {
    const int k = (int)(s % K);
    const int group = (int)std::min<int64_t>(K, n - (s - k));  // steps drawn with this one
    const int64_t off = in_graph ? s : -1;
    if (group >= kDrawGroup && k == 0) {
      const int r = c->prec == UASD_FP64 ? draw_ahead<double>(c, group, off)
                                         : draw_ahead<float>(c, group, off);
      if (r) return r;
    }
    if (int r = llg_step(c, alg, off, group >= kDrawGroup ? k : -1)) return r;
    if (!in_graph) c->step += 1;
  }
  return UASD_OK;
}

// Whether n more steps (kind 0) or sweeps (kind 1) of a call should be
// replayed as graphs although none were asked for: the launches are short
// (items = sites x ensembles of one), the program has already launched `after`
// of them one by one with nothing changed in between, and nobody is timing the
// kernels or capturing the stream.  A replayed launch of a small lattice is
// 0.4-1.6 us shorter than an enqueued one (its arguments already lie in device
// memory): 432 sites, 14 neighbours, FP64 13.3 -> 10.3 us a step, FP32 11.9 ->
// 8.6; 16,000 sites 14.3 -> 11.7; 65,536 sites (film) FP32 14.8 -> 13.0, FP64
// 16.7 -> 15.6; nothing from 2^18 items on.  Building a graph costs 3.3 us a
// launch (430 us for 64 steps) and the process's first 3.6 ms more, which 2048
// steps or 512 sweeps would have repaid, hence `after`.
bool repeats_pay(uasd_ctx *c, int kind, int alg, uint64_t seed, int64_t items, int64_t n,
                 int64_t after) {
  if (c->graph_steps > 0 || c->timing || c->replays_off || items > 131072) return false;
  if (!stream_free(c)) return false;
  if (c->repeats.size() > 64) c->repeats.clear();
  auto &r = c->repeats[std::make_tuple(kind, alg, seed)];
  if (r.first != c->gen) r = {c->gen, 0};
  r.second += n;
  return r.second - n >= after;
}

// nsteps steps in resident launches.
template <typename R>
int llg_resident_steps(uasd_ctx *c, int alg, int64_t nsteps) {
  const bool philox = llg_view<R>(c).noise_mode == UASD_NOISE_PHILOX;
  const int64_t chunk = resident_steps(c);
  for (int64_t s = 0; s < nsteps; s += chunk) {
    const int n = (int)std::min(chunk, nsteps - s);
    // a single step: its draw and the resident launch take longer than the
    // two half steps (432 sites FP64 14.7 against 11.8 us, FP32 12.5 against
    // 10.4); two steps are faster (10.3, 8.4)
    if (philox && n == 1) return llg_steps(c, alg, 1, false);
    if (philox)
      if (int r = draw_ahead<R>(c, n, -1)) return r;
    uasd::LLGDev<R> prm = llg_view<R>(c);
    if (philox) prm.nsave = quads<R>(c, c->nsave);
    HIP_TRY(uasd::launch_llg_resident<R>(c->stream, alg, ham_view<R>(c), prm, c->lres.dev, n,
                                         (size_t)c->lds_max, quads<R>(c, c->spins, 0)));
    count(c, UASD_LAUNCH_LLG_RESIDENT);
    c->step += (uint64_t)n;
  }
  return UASD_OK;
}

int sd_steps_run(uasd_ctx *c, int alg, int64_t nsteps) {
  const bool open = stream_free(c);  // not in a caller's own capture, which takes no tables
  if (open)
    if (int r = build_llg_resident(c)) return r;
  if (open && llg_use_resident(c))
    return c->prec == UASD_FP64 ? llg_resident_steps<double>(c, alg, nsteps)
                                : llg_resident_steps<float>(c, alg, nsteps);
  int64_t s = 0;
  auto replay = [&](int K) -> int {
    auto body = [&]() -> int {
      if (int r = llg_steps(c, alg, K, true)) return r;
      HIP_TRY(uasd::launch_counter(queue(c), 0, c->ctr.as<uint64_t>(), (uint64_t)K, 1));
      return UASD_OK;
    };
    for (; nsteps - s >= K; s += K)
      if (int r = replay_graph(c, std::make_tuple(0, alg, K, (uint64_t)0), 0, c->step, K, 4, body))
        return r;
    return UASD_OK;
  };
  if (c->graph_steps > 0) {
    if (int r = replay(c->graph_steps)) return r;
  } else if (repeats_pay(c, 0, alg, 0, (int64_t)c->N * c->M, nsteps, 2048)) {
    for (int K : {64, 16})
      if (replay(K)) {
        replay_failed(c);
        break;
      }
  }
  return llg_steps(c, alg, nsteps - s, false);
}

}  // namespace

extern "C" {

int uasd_effective_field(uasd_ctx *c, double *beff, double *energy) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_ex || !c->have_state) return fail(UASD_ERR_STATE, "exchange or moments not set");
  if (int r = rebuild_classes(c)) return r;
  int r = c->prec == UASD_FP64
              ? run_field<double>(c, false, energy != nullptr, false, beff != nullptr)
              : run_field<float>(c, false, energy != nullptr, false, beff != nullptr);
  if (r) return r;
  HostIo io(c);
  if (beff && (r = download_vec(io, c->field, 0, beff, false))) return r;
  if (energy) {
    std::vector<double> red;
    r = c->prec == UASD_FP64 ? reduce_moments<double>(c, true, false, red)
                             : reduce_moments<float>(c, true, false, red);
    if (r) return r;
    double e = 0.0;
    for (int k = 0; k < c->M; ++k) e += red[4 * (size_t)k + 3];
    *energy = e * uasd::kMub / uasd::kMry;
  }
  return io.wait();
}

// Builds c->res for the current lists, classes and colouring.
static int build_resident(uasd_ctx *c) {
  auto &r = c->res;
  if (r.cls_version == c->cls_version && r.col_version == c->col_version) return UASD_OK;
  r.ok = false;
  r.cls_version = c->cls_version;
  r.col_version = c->col_version;
  const int N = c->N, ncol = c->ncolors;
  // the limits that need no look at the lists, or at a few bonds only, first
  if ((int64_t)N * c->M > (int64_t)ncol << 18) return UASD_OK;
  const size_t lds0 = uasd::res_lds_spins(c->rsize, 0);
  const size_t most = std::min<size_t>(
      (size_t)uasd::kResThreads * ncol,
      ((size_t)c->lds_max - lds0) / (uasd::res_lds_spins(c->rsize, 1) - lds0));
  if (bond_spans(c, (int)most)) return UASD_OK;
  const std::vector<int> off = independent_ranges(c);
  const int ncomp = (int)off.size() - 1;
  int nmax = 0;
  for (int k = 0; k < ncomp; ++k) nmax = std::max(nmax, off[k + 1] - off[k]);
  if (uasd::res_lds_spins(c->rsize, nmax) > (size_t)c->lds_max || nmax > 65536) return UASD_OK;
  std::vector<int> ptr((size_t)ncomp * (ncol + 1)), pos(N);
  std::vector<int> site(N);
  int cmax = 1;
  for (int k = 0; k < ncomp; ++k) {
    int *pc = ptr.data() + (size_t)k * (ncol + 1);
    for (int i = off[k]; i < off[k + 1]; ++i) pc[c->color_of_site[i] + 1]++;
    for (int q = 1; q <= ncol; ++q) {
      cmax = std::max(cmax, pc[q]);
      pc[q] += pc[q - 1];
    }
    std::vector<int> at(pc, pc + ncol);
    for (int i = off[k]; i < off[k + 1]; ++i) {
      pos[i] = at[c->color_of_site[i]]++;
      site[off[k] + pos[i]] = i;
    }
  }
  const int W = c->W, Wd = c->Wd;
  std::vector<uint16_t> nb((size_t)(W + Wd) * N);
  auto fill = [&](const std::vector<int> &list, int w, uint16_t *out) {
    for (int k = 0; k < ncomp; ++k)
      for (int p = off[k]; p < off[k + 1]; ++p)
        for (int j = 0; j < w; ++j) out[(size_t)j * N + p] = (uint16_t)pos[list[(size_t)j * N + site[p]]];
  };
  fill(c->nbr_host, W, nb.data());
  fill(c->dnbr_host, Wd, nb.data() + (size_t)W * N);
  std::vector<uasd::SiteClass> cls(N);
  for (int p = 0; p < N; ++p) {
    const int i = site[p];
    cls[p] = uasd::SiteClass{c->ex_row_of_site.empty() ? 0 : c->ex_row_of_site[i],
                             c->dm_row_of_site.empty() ? -1 : c->dm_row_of_site[i],
                             c->an_row_of_site.empty() ? -1 : c->an_row_of_site[i], 0};
  }
  // one allocation: classes, offsets, colour pointers, sites, lists
  std::vector<char> all;
  auto put = [&](const void *p, size_t n) {
    const size_t at = all.size();
    all.resize(at + (n + 15) / 16 * 16);
    std::memcpy(all.data() + at, p, n);
    return at;
  };
  const size_t ocls = put(cls.data(), cls.size() * sizeof(cls[0])),
               ooff = put(off.data(), off.size() * sizeof(int)),
               optr = put(ptr.data(), ptr.size() * sizeof(int)),
               osite = put(site.data(), site.size() * sizeof(int)),
               onb = put(nb.data(), nb.size() * sizeof(uint16_t));
  if (upload_raw(c, r.buf, all)) {  // no room for tables that the launched kernels do not need
    (void)hipGetLastError();
    return UASD_OK;
  }
  const char *base = r.buf.as<char>();
  r.dev = uasd::ResDev{ncomp,
                       ncol,
                       nmax,
                       cmax,
                       reinterpret_cast<const int *>(base + ooff),
                       reinterpret_cast<const int *>(base + optr),
                       reinterpret_cast<const int *>(base + osite),
                       reinterpret_cast<const uasd::SiteClass *>(base + ocls),
                       reinterpret_cast<const uint16_t *>(base + onb),
                       reinterpret_cast<const uint16_t *>(base + onb) + (size_t)W * N};
  r.ncomp = ncomp;
  r.nmax = nmax;
  r.waves = 0;
  const int slots = (std::min(cmax, uasd::kResThreads) + 63) / 64;
  for (int k = 0; k < ncomp; ++k)
    for (int q = 0; q < ncol; ++q) {
      const int *pc = ptr.data() + (size_t)k * (ncol + 1) + q;
      r.waves += uasd::res_waves(pc[1] - pc[0], slots);
    }
  r.ok = true;
  c->gen += 1;  // captured sweeps hold the old tables
  return UASD_OK;
}

// Uploads the per-ensemble MC constants and the colour lists and fills mp.
static int mc_prepare(uasd_ctx *c, char mode, const double *temps, uint64_t seed,
                      uasd::MCParams &mp) {
  if (mode != 'M' && mode != 'H') return fail(UASD_ERR_UNSUPPORTED, "mode must be 'M' or 'H'");
  if (!temps) return fail(UASD_ERR_ARG, "temps is null");
  if (!c->have_ex || !c->have_state) return fail(UASD_ERR_STATE, "exchange or moments not set");
  if (c->ext_mode == 2)
    return fail(UASD_ERR_UNSUPPORTED, "MC takes a uniform external field (as mc_evolve's extfield)");
  if (int r = rebuild_classes(c)) return r;
  if (int r = build_coloring(c)) return r;
  if (int r = build_resident(c)) return r;
  const int M = c->M;
  for (int k = 0; k < M; ++k)
    if (!(temps[k] > 0.0)) return fail(UASD_ERR_ARG, "MC temperatures must be > 0");
  // per-ensemble constants (montecarlo.f90:141, montecarlo_common.f90:190, 397)
  std::vector<double> host(6 * (size_t)M);
  for (int k = 0; k < M; ++k) {
    host[k] = (double)(2.0f / 25.0f) * std::pow(uasd::kKBolt * temps[k] / uasd::kMub, 0.20);
    host[M + k] = 1.0 / uasd::kKBolt / (c->temprescale * temps[k] + 1.0e-15);
    host[2 * (size_t)M + k] = 1.0 / uasd::kKBolt / (c->temprescale * temps[k]);
  }
  for (int k = 0; k < M; ++k)
    for (int d = 0; d < 3; ++d)
      host[3 * (size_t)M + 3 * k + d] = c->ext_u_host.empty() ? 0.0 : c->ext_u_host[3 * k + d];
  const size_t cbytes = host.size() * sizeof(double);
  HIP_TRY(c->mcbuf.ensure(cbytes + c->color_sites.size() * sizeof(int)));
  HIP_TRY(hipMemcpyAsync(c->mcbuf.p, host.data(), cbytes, hipMemcpyHostToDevice, c->stream));
  int *sites_dev = reinterpret_cast<int *>(static_cast<char *>(c->mcbuf.p) + cbytes);
  HIP_TRY(hipMemcpyAsync(sites_dev, c->color_sites.data(), c->color_sites.size() * sizeof(int),
                         hipMemcpyHostToDevice, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  mp = uasd::MCParams{};
  const double *base = c->mcbuf.as<double>();
  mp.sites = sites_dev;
  mp.delta = base;
  mp.beta = base + M;
  mp.hbeta = base + 2 * (size_t)M;
  mp.ext = base + 3 * (size_t)M;
  mp.seed = seed;
  mp.heat_bath = mode == 'H';
  return UASD_OK;
}

// Whether the sweeps run in k_mc_resident: systems that fit in LDS, whose
// colours hold no more sites on average than its workgroup has threads, and
// few enough updates per colour that a launch of them is mostly launch.
//  - Sites per colour: a colour costs 1.4-2.2 us (14 neighbours) against 5-7
//    us for its launch; with more sites than threads the one CU needs longer
//    for a phase than the whole chip for a launch.  Per sweep, launches ->
//    resident, 14 neighbours: 432 sites FP64 54 -> 18 us (FP32 40 -> 13), 2000
//    sites 63 -> 27 (44 -> 17), heat bath 57 -> 26, 4394 sites (10 colours,
//    439 sites each) 77 -> 47.
//  - Updates per colour: 2^18 of them take the launch path 6-17 us.  At 228k
//    (1024 ensembles of 2000 sites, 9 colours) 158 -> 113 us a sweep, at 262k
//    (alloy pairs of 1024 sites, 256 ensembles, 2 colours) 29 -> 21 us; at
//    600k (64 alloys, 32 ensembles) 54 -> 61 us, slower.
//  - Fewer than 3000 idle wavefronts a phase (9000 in FP32 Metropolis with its
//    cheap moves): a phase of resident launches is 1.7 us and 0.8 ns a wavefront
//    longer, a launched colour 4-5 us and 16 ns per 1000 updates, 1.0 ns a full
//    wavefront.  Heat bath FP64, launches against resident, sites x systems, idle
//    wavefronts in brackets: 16 x 1024 (864) 8.2 -> 5.3 us a sweep, 256 x 2048
//    (none) 16.7 -> 12.1, 64 x 8192 (3072) 16.7 -> 17.3, 4 x 4096 (3936) 8.2 ->
//    9.7, 2 x 262,144 16.2 -> 457; FP32 Metropolis 64 x 8192 12.2 -> 7.9, 2 x 8192
//    (8032) 7.7 -> 6.7, 16 x 32,768 (27,648) 12.3 -> 23.7.
// Not where a launch shape was asked for: it is one of the colour pass.
static bool mc_can_be_resident(const uasd_ctx *c, bool heat_bath) {
  if (!c->res.ok || c->res.nmax > uasd::kResThreads * c->ncolors) return false;
  const int64_t items = (int64_t)c->N * c->M, col = c->ncolors;
  const double idle = uasd::res_idle_waves(c->res.waves * c->M / col, items / col, 1.25);
  return items <= col << 18 && idle < (c->prec == UASD_FP32 && !heat_bath ? 9000 : 3000);
}

static bool mc_use_resident(const uasd_ctx *c, bool heat_bath) {
  return mc_can_be_resident(c, heat_bath) && c->tune[2].chosen != uasd::kShapeAsked;
}

// nsweeps sweeps in resident launches of at most kResSweeps, from mp.sweep on.
// The predicted moments (quad array 1), which every LLG step writes before it
// reads them, lend their memory to the trial moves.
static int mc_resident(uasd_ctx *c, uasd::MCParams mp, int64_t nsweeps) {
  constexpr int64_t kResSweeps = 1024;
  for (int64_t s = 0; s < nsweeps; s += kResSweeps) {
    const int n = (int)std::min(kResSweeps, nsweeps - s);
    tic(c, 3);
    if (c->prec == UASD_FP64)
      HIP_TRY(uasd::launch_mc_resident<double>(queue(c), ham_view<double>(c), mp, c->res.dev, n,
                                               (size_t)c->lds_max, quads<double>(c, c->spins, 0),
                                               quads<double>(c, c->spins, 1)));
    else
      HIP_TRY(uasd::launch_mc_resident<float>(queue(c), ham_view<float>(c), mp, c->res.dev, n,
                                              (size_t)c->lds_max, quads<float>(c, c->spins, 0),
                                               quads<float>(c, c->spins, 1)));
    count(c, UASD_LAUNCH_MC_RESIDENT);
    if (int r = toc(c, 3)) return r;
    mp.sweep += (uint64_t)n;
  }
  return UASD_OK;
}

// Launch shape of a colour of nsites sites.
static uasd::Tune mc_tune(const uasd_ctx *c, int nsites) {
  return uasd::default_tune(c->tune[2], (int64_t)nsites * c->M, c->W);
}

// nsweeps colour-ordered sweeps; every launch is asynchronous on the stream.
static int mc_run(uasd_ctx *c, uasd::MCParams mp, int64_t nsweeps) {
  const int *sites_dev = mp.sites;
  if (mc_use_resident(c, mp.heat_bath)) {
    mp.sweep = c->mc_sweep;
    if (int r = mc_resident(c, mp, nsweeps)) return r;
    c->mc_sweep += (uint64_t)nsweeps;
    return UASD_OK;
  }
  for (int64_t s = 0; s < nsweeps; ++s) {
    mp.sweep = c->mc_sweep;
    for (int col = 0; col < c->ncolors; ++col) {
      mp.sites = sites_dev + c->color_ptr[col];
      mp.nsites = c->color_ptr[col + 1] - c->color_ptr[col];
      mp.site0 = c->color_start[col];
      mp.sstride = c->color_stride[col];
      tic(c, 3);
      if (c->prec == UASD_FP64) {
        HIP_TRY(uasd::launch_mc<double>(queue(c), mc_tune(c, mp.nsites), ham_view<double>(c), mp,
                                        quads<double>(c, c->spins, 0)));
      } else {
        HIP_TRY(uasd::launch_mc<float>(queue(c), mc_tune(c, mp.nsites), ham_view<float>(c), mp,
                                       quads<float>(c, c->spins, 0)));
      }
      count(c, UASD_LAUNCH_MC_COLOUR);
      if (int r = toc(c, 3)) return r;
    }
    c->mc_sweep += 1;
  }
  return UASD_OK;
}

int uasd_mc_sweeps(uasd_ctx *c, char mode, const double *temps, int64_t nsweeps, uint64_t seed) {
  if (int r = check_ctx(c)) return r;
  if (nsweeps < 0) return fail(UASD_ERR_ARG, "nsweeps < 0");
  uasd::MCParams mp;
  if (int r = mc_prepare(c, mode, temps, seed, mp)) return r;
  if (int r = region_tic(c)) return r;
  if (int r = mc_sweeps_run(c, mode, mp, nsweeps, seed)) return r;
  return region_toc(c);
}

}  // extern "C"

namespace {

int mc_sweeps_run(uasd_ctx *c, char mode, const uasd::MCParams &mp, int64_t nsweeps,
                  uint64_t seed) {
  int64_t s = 0;
  auto replay = [&](int K) -> int {
    auto body = [&]() -> int {
      uasd::MCParams g = mp;
      g.sweep_dev = c->ctr.as<uint64_t>() + 1;
      const bool resident = mc_use_resident(c, mp.heat_bath);
      if (resident) {
        g.sweep = 0;
        if (int r = mc_resident(c, g, K)) return r;
      }
      for (int j = 0; j < K && !resident; ++j) {
        g.sweep = (uint64_t)j;
        for (int col = 0; col < c->ncolors; ++col) {
          g.sites = mp.sites + c->color_ptr[col];
          g.nsites = c->color_ptr[col + 1] - c->color_ptr[col];
          g.site0 = c->color_start[col];
          g.sstride = c->color_stride[col];
          if (c->prec == UASD_FP64) {
            HIP_TRY(uasd::launch_mc<double>(queue(c), mc_tune(c, g.nsites), ham_view<double>(c), g,
                                            quads<double>(c, c->spins, 0)));
          } else {
            HIP_TRY(uasd::launch_mc<float>(queue(c), mc_tune(c, g.nsites), ham_view<float>(c), g,
                                           quads<float>(c, c->spins, 0)));
          }
        }
      }
      HIP_TRY(uasd::launch_counter(queue(c), 1, c->ctr.as<uint64_t>(), (uint64_t)K, 1));
      return UASD_OK;
    };
    for (; nsweeps - s >= K; s += K)
      if (int r = replay_graph(c, std::make_tuple(1, (int)mode, K, seed), 1, c->mc_sweep, K, 5,
                               body))
        return r;
    return UASD_OK;
  };
  if (c->graph_steps > 0) {
    if (int r = replay(c->graph_steps)) return r;
  } else if (!mc_use_resident(c, mp.heat_bath) &&
             repeats_pay(c, 1, mode, seed, (int64_t)c->N * c->M / std::max(c->ncolors, 1),
                         nsweeps, 512)) {
    for (int K : {16, 4})
      if (replay(K)) {
        replay_failed(c);
        break;
      }
  }
  return mc_run(c, mp, nsweeps - s);
}

}  // namespace

extern "C" {

// ---------------------------------------------------------------- tuning
int uasd_index_bytes(uasd_ctx *c, int *exchange, int *dm) {
  if (int r = check_ctx(c)) return r;
  const bool i32 = c->tune[0].idx32 != 0;  // as the LLG kernels are tuned
  if (exchange) *exchange = c->use16 && !i32 ? 2 : 4;
  if (dm) *dm = c->use16_dm && !i32 ? 2 : 4;
  return UASD_OK;
}

int uasd_llg_tile(uasd_ctx *c, int *tile) {
  if (int r = check_ctx(c)) return r;
  if (!tile) return fail(UASD_ERR_ARG, "tile must not be NULL");
  *tile = llg_use_resident(c) ? 0 : launched_tile(c);
  return UASD_OK;
}

int uasd_launch_counts(uasd_ctx *c, int64_t *counts) {
  if (int r = check_ctx(c)) return r;
  if (!counts) return fail(UASD_ERR_ARG, "counts must not be NULL");
  std::copy(c->launches, c->launches + UASD_NUM_LAUNCH_KINDS, counts);
  return UASD_OK;
}

int uasd_set_tuning(uasd_ctx *c, int kind, int gather, int block) {
  if (int r = check_ctx(c)) return r;
  c->gen += 1;
  if (kind < 0 || kind > 2) return fail(UASD_ERR_ARG, "kind must be 0 (LLG), 1 (field) or 2 (MC)");
  // block may carry flags: 0x10000 non-temporal list loads, 0x20000 int32
  // entries, (k << 18) LDS-tiled stencil shape k and 0x400000 resident
  // workgroups looping over tiles (LLG only), 0x800000 a separate DM gather
  // where the DM bonds are the exchange bonds (context-wide), 0x1000000 two
  // adjacent ensembles per thread (MC only)
  uasd::Tune t{gather, block & 0xffff, (block >> 16) & 1, (block >> 17) & 1, (block >> 18) & 0xf,
               (block >> 22) & 1, (block >> 24) & 1, uasd::kShapeAsked};
  if (!uasd::tune_valid(t) || (block >> 25) != 0 || (kind != 0 && t.tile != 0) ||
      (kind != 2 && t.pair != 0))
    return fail(UASD_ERR_ARG, "gather must be 2, 4, 8 or 16 and block 64, 128 or 256");
  c->tune[kind] = t;
  c->tune_no_fuse = ((block >> 23) & 1) != 0;
  return UASD_OK;
}

int uasd_get_tuning(uasd_ctx *c, int kind, int *gather, int *block) {
  if (int r = check_ctx(c)) return r;
  if (kind < 0 || kind > 2) return fail(UASD_ERR_ARG, "kind must be 0 (LLG), 1 (field) or 2 (MC)");
  // the shape that is launched (colours differ in size: that of an average one)
  const int64_t items = (int64_t)c->N * c->M / (kind == 2 ? std::max(c->ncolors, 1) : 1);
  const uasd::Tune t = uasd::default_tune(c->tune[kind], items, c->W);
  if (gather) *gather = t.gather;
  if (block)
    *block = t.block | (t.nt << 16) | (t.idx32 << 17) | (t.tile << 18) | (t.pipe << 22) |
             ((c->tune_no_fuse ? 1 : 0) << 23) | (t.pair << 24);
  return UASD_OK;
}

}  // extern "C"

namespace {

// Copies of the spin quads and the counters, restored after a tuning run so
// that tuning leaves the trajectory untouched.
struct StateGuard {
  uasd_ctx *c;
  DevBuf save;
  uint64_t step, sweep;
  bool timing;
  int err = UASD_OK;
  explicit StateGuard(uasd_ctx *cc) : c(cc), step(cc->step), sweep(cc->mc_sweep), timing(cc->timing) {
    const size_t n = 3 * quad_bytes(c);
    hipError_t e = save.ensure(n);
    if (e == hipSuccess) e = hipMemcpyAsync(save.p, c->spins.p, n, hipMemcpyDeviceToDevice, c->stream);
    if (e != hipSuccess) err = fail(UASD_ERR_HIP, std::string("tuning state copy: ") + hipGetErrorString(e));
    c->timing = false;
  }
  int restore() {
    const size_t n = 3 * quad_bytes(c);
    HIP_TRY(hipMemcpyAsync(c->spins.p, save.p, n, hipMemcpyDeviceToDevice, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    c->step = step;
    c->mc_sweep = sweep;
    c->timing = timing;
    return UASD_OK;
  }
};

struct EventPair {
  hipEvent_t a = nullptr, b = nullptr;
  ~EventPair() {
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
  }
};

// ------------------------------------------------------ autotuner cache
// Winners of uasd_autotune_* per workload, kept for the process once
// uasd_set_tune_cache has switched the cache on, and read from / appended to
// its text file when it names one: one line per workload, "key gather block
// nt idx32 tile pipe best_ms".  The key holds what the launch shapes' speed
// depends on: the kernel family, solver or mode, precision, sizes, list
// widths, terms, site order, lattice dimensions, list entry width, noise
// source (none at a uniform T = 0) and kTuneKernels.
std::mutex g_tune_mu;
bool g_tune_on = false;
std::string g_tune_path;
std::map<std::string, std::pair<uasd::Tune, double>> g_tune;

// kTuneKernels is the generation of the kernels that were timed: entries of an
// earlier one (none in the key: 1) are times and winners of other code, and
// some of its small systems' were those of a path that ignored the shape.
constexpr int kTuneKernels = 2;

std::string tune_key(const uasd_ctx *c, const char *kind, int alg) {
  char buf[320];
  std::snprintf(buf, sizeof buf,
                "v2/gfx950/%s/a%d/%s/N%d/M%d/seg%d/W%d/Wd%d/an%d/ext%d/order%d/lat%d,%d,%d,%d/i16%d%d/"
                "noise%d/k%d",
                kind, alg, c->prec == UASD_FP64 ? "fp64" : "fp32", c->N, c->M, c->nseg, c->W,
                c->Wd, c->an_rows > 0 ? 1 : 0, c->ext_mode, c->order_na, c->lat_na, c->lat_n1,
                c->lat_n2, c->lat_n3, c->use16 ? 1 : 0, c->use16_dm ? 1 : 0,
                c->temp_uniform && c->temp0 == 0.0 ? 0 : c->noise_mode, kTuneKernels);
  return buf;
}

bool tune_lookup(const std::string &key, uasd::Tune &t, double &ms) {
  std::lock_guard<std::mutex> lock(g_tune_mu);
  if (!g_tune_on) return false;
  auto it = g_tune.find(key);
  if (it == g_tune.end()) return false;
  t = it->second.first;
  ms = it->second.second;
  return true;
}

void tune_store(const std::string &key, const uasd::Tune &t, double ms) {
  std::lock_guard<std::mutex> lock(g_tune_mu);
  if (!g_tune_on) return;
  g_tune[key] = {t, ms};
  if (g_tune_path.empty()) return;
  if (FILE *f = std::fopen(g_tune_path.c_str(), "a")) {
    std::fprintf(f, "%s %d %d %d %d %d %d %d %.6f\n", key.c_str(), t.gather, t.block, t.nt,
                 t.idx32, t.tile, t.pipe, t.pair, ms);
    std::fclose(f);
  }
}

// Key of a context whose steps or sweeps could be resident: its entry also
// says whether that was faster than every shape, which other contexts of the
// same sizes (other bonds) must not take over.
std::string resident_key(const std::string &key, bool won) { return key + (won ? "/res1" : "/res0"); }

// The kept result of this workload into slot, as tune_search leaves it.
bool tune_cached(const std::string &key, bool resident, uasd::Tune *slot, double &ms) {
  uasd::Tune t;
  bool won = resident;
  if (!resident) {
    if (!tune_lookup(key, t, ms)) return false;
  } else if (!tune_lookup(resident_key(key, true), t, ms)) {
    won = false;
    if (!tune_lookup(resident_key(key, false), t, ms)) return false;
  }
  if (!uasd::tune_valid(t)) return false;
  t.chosen = won ? uasd::kShapeResident : uasd::kShapeAsked;
  *slot = t;
  return true;
}

void tune_keep(const std::string &key, bool resident, const uasd::Tune &t, double ms) {
  tune_store(resident ? resident_key(key, t.chosen == uasd::kShapeResident) : key, t, ms);
}

// Times run(n), n steps or sweeps in asynchronous launches on c->stream, for
// every shape and leaves the fastest in *slot, marked as asked for.  pair: also
// two ensembles per thread (the MC colour pass, M even); resident: also the
// resident launch, which run() makes while the slot is marked kShapeResident.
// Its systems and lists are loaded once a call, so it is timed in calls of
// kResidentCall, as programs make them; the slot then keeps that mark beside
// the fastest shape unless a shape was faster by a tenth, more than two
// searches differ.  Alloy batch of 10 systems, 32 temperatures, timed over one
// sweep: launched, 18.4 us a sweep of a 20-sweep call; resident 14.0.
template <typename Run>
int tune_search(uasd_ctx *c, uasd::Tune *slot, int n, Run &&run, double *best_ms, bool pair,
                bool resident) {
  EventPair ev;
  HIP_TRY(hipEventCreate(&ev.a));
  HIP_TRY(hipEventCreate(&ev.b));
  const int gathers[] = {2, 4, 8, 16};
  const int blocks[] = {64, 128, 256};
  std::vector<uasd::Tune> cand;
  const int nidx = c->use16 || c->use16_dm ? 2 : 1;
  for (int ix = 0; ix < nidx; ++ix)
    for (int nt = 0; nt < 2; ++nt)
      for (int g : gathers)
        for (int bl : blocks) {
          cand.push_back(uasd::Tune{g, bl, nt, ix, 0});
          if (pair && c->M % 2 == 0) cand.push_back(uasd::Tune{g, bl, nt, ix, 0, 0, 1});
        }
  if (slot == &c->tune[0]) {
    build_stencil(c);
    for (int k = 1; k <= uasd::kNumTileShapes; ++k)
      if (tile_fits(c, k))
        for (int pipe = 0; pipe < 2; ++pipe) cand.push_back(uasd::Tune{4, 256, 0, 0, k, pipe});
  }
  // one timed run each, then the fastest few again over several runs: a single
  // run of a small lattice (tens of us) ranks shapes within its own scatter
  auto timed = [&](const uasd::Tune &cd, int call, int reps, float &ms) -> int {
    *slot = cd;
    if (int r = run(call)) return r;
    HIP_TRY(hipEventRecord(ev.a, c->stream));
    for (int k = 0; k < reps; ++k)
      if (int r = run(call)) return r;
    HIP_TRY(hipEventRecord(ev.b, c->stream));
    HIP_TRY(hipEventSynchronize(ev.b));
    HIP_TRY(hipEventElapsedTime(&ms, ev.a, ev.b));
    ms *= (float)n / ((float)reps * (float)call);
    return UASD_OK;
  };
  std::vector<std::pair<float, int>> rank;
  for (size_t i = 0; i < cand.size(); ++i) {
    float ms = 0.f;
    cand[i].chosen = uasd::kShapeAsked;
    if (int r = timed(cand[i], n, 1, ms)) return r;
    rank.emplace_back(ms, (int)i);
  }
  std::sort(rank.begin(), rank.end());
  constexpr int kFinal = 5, kReps = 6, kResidentCall = 64;
  uasd::Tune best = cand[rank[0].second];
  float best_t = 1e30f;
  for (int k = 0; k < kFinal && k < (int)rank.size(); ++k) {
    float ms = 0.f;
    if (int r = timed(cand[rank[k].second], n, kReps, ms)) return r;
    if (ms < best_t) {
      best_t = ms;
      best = *slot;
    }
  }
  if (resident) {
    uasd::Tune res = best;
    res.chosen = uasd::kShapeResident;
    float ms = 0.f;
    if (int r = timed(res, kResidentCall, 2, ms)) return r;
    if (ms < 1.1f * best_t) {
      best_t = ms;
      best = res;
    }
  }
  *slot = best;
  if (best_ms) *best_ms = best_t;
  return UASD_OK;
}

}  // namespace

extern "C" {

int uasd_autotune_llg(uasd_ctx *c, int alg, int steps, double *best_ms) {
  if (int r = check_ctx(c)) return r;
  if (!sde_supported(alg))
    return fail(UASD_ERR_UNSUPPORTED, "SDEalgh must be 1 (midpoint), 4 (Heun), 5 (Depondt), 6 (SIB) or 7 (spherical midpoint)");
  if (steps <= 0) return fail(UASD_ERR_ARG, "steps must be > 0");
  if (int r = ready_for_llg(c)) return r;
  build_stencil(c);
  if (int r = build_llg_resident(c)) return r;
  const std::string key = tune_key(c, "llg", alg);
  const bool resident = llg_can_be_resident(c);
  uasd::Tune cached;
  double cached_ms = 0.0;
  if (tune_cached(key, resident, &cached, cached_ms) && cached.pair == 0 &&
      (cached.tile == 0 || tile_fits(c, cached.tile))) {
    c->tune[0] = c->tune[1] = cached;
    c->tune[1].tile = c->tune[1].pipe = 0;
    if (best_ms) *best_ms = cached_ms;
    c->gen += 1;
    return UASD_OK;
  }
  StateGuard g(c);
  if (g.err) return g.err;
  double ms_found = 0.0;
  int r = tune_search(c, &c->tune[0], steps, [&](int n) -> int {
    if (!llg_use_resident(c)) return llg_steps(c, alg, n, false);
    return c->prec == UASD_FP64 ? llg_resident_steps<double>(c, alg, n)
                                : llg_resident_steps<float>(c, alg, n);
  }, &ms_found, false, resident);
  if (r) return r;
  if (best_ms) *best_ms = ms_found;
  tune_keep(key, resident, c->tune[0], ms_found);
  c->tune[1] = c->tune[0];  // the field kernel gathers the same way
  c->gen += 1;
  return g.restore();
}

int uasd_autotune_mc(uasd_ctx *c, char mode, const double *temps, int sweeps, double *best_ms) {
  if (int r = check_ctx(c)) return r;
  if (sweeps <= 0) return fail(UASD_ERR_ARG, "sweeps must be > 0");
  uasd::MCParams mp;
  if (int r = mc_prepare(c, mode, temps, 0x7u, mp)) return r;
  const std::string key = tune_key(c, "mc", (int)mode);
  const bool resident = mc_can_be_resident(c, mp.heat_bath);
  uasd::Tune cached;
  double cached_ms = 0.0;
  if (tune_cached(key, resident, &cached, cached_ms) && cached.tile == 0) {
    c->tune[2] = cached;
    if (best_ms) *best_ms = cached_ms;
    c->gen += 1;
    return UASD_OK;
  }
  StateGuard g(c);
  if (g.err) return g.err;
  double ms_found = 0.0;
  int r = tune_search(c, &c->tune[2], sweeps, [&](int n) -> int { return mc_run(c, mp, n); },
                      &ms_found, true, resident);
  if (r) return r;
  if (best_ms) *best_ms = ms_found;
  tune_keep(key, resident, c->tune[2], ms_found);
  c->gen += 1;
  return g.restore();
}

int uasd_set_tune_cache(int enable, const char *path) {
  std::lock_guard<std::mutex> lock(g_tune_mu);
  g_tune_on = enable != 0;
  g_tune_path = (enable && path) ? path : "";
  if (!g_tune_on) {
    g_tune.clear();
    return UASD_OK;
  }
  if (g_tune_path.empty()) return UASD_OK;
  FILE *f = std::fopen(g_tune_path.c_str(), "r");
  if (!f) return UASD_OK;  // a new file: created by the first result
  char key[320];
  uasd::Tune t;
  double ms = 0.0;
  int loaded = 0;
  while (std::fscanf(f, "%319s %d %d %d %d %d %d %d %lf", key, &t.gather, &t.block, &t.nt,
                     &t.idx32, &t.tile, &t.pipe, &t.pair, &ms) == 9) {
    if (uasd::tune_valid(t)) {
      g_tune[key] = {t, ms};
      ++loaded;
    }
  }
  std::fclose(f);
  (void)loaded;
  return UASD_OK;
}

int uasd_measure(uasd_ctx *c, double *msum, double *energy) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_state) return fail(UASD_ERR_STATE, "moments not set");
  if (!msum) return fail(UASD_ERR_ARG, "msum is null");
  if (energy) {
    if (!c->have_ex) return fail(UASD_ERR_STATE, "exchange not set");
    if (int r = rebuild_classes(c)) return r;
    int r = c->prec == UASD_FP64 ? run_field<double>(c, false, true, false, false)
                                 : run_field<float>(c, false, true, false, false);
    if (r) return r;
  }
  std::vector<double> red;
  int r = c->prec == UASD_FP64 ? reduce_moments<double>(c, energy != nullptr, false, red)
                               : reduce_moments<float>(c, energy != nullptr, false, red);
  if (r) return r;
  const int nv = energy ? 4 : 3;
  for (int k = 0; k < c->M; ++k) {
    for (int d = 0; d < 3; ++d) msum[3 * k + d] = red[(size_t)nv * k + d];
    if (energy) energy[k] = red[(size_t)nv * k + 3] * uasd::kMub / uasd::kMry;
  }
  return UASD_OK;
}

int uasd_set_site_order(uasd_ctx *c, int na) {
  if (int r = check_ctx(c)) return r;
  if (na < 1 || c->N % na != 0) return fail(UASD_ERR_ARG, "na must be >= 1 and divide natom");
  if (c->have_ex || c->have_state || c->have_llg || c->Wd > 0 || c->an_rows > 0 || c->ext_mode == 2)
    return fail(UASD_ERR_STATE, "set the site order before any Hamiltonian, moment or LLG upload");
  if (c->nseg > 1 && na > 1) return fail(UASD_ERR_UNSUPPORTED, "site order with several segments");
  c->order_na = na;
  c->order_nc = c->N / na;
  c->gen += 1;
  return UASD_OK;
}

int uasd_set_lattice_dims(uasd_ctx *c, int na, int n1, int n2, int n3) {
  if (int r = check_ctx(c)) return r;
  if (na == 0 && n1 == 0 && n2 == 0 && n3 == 0) {  // forget the lattice
    c->lat_na = c->lat_n1 = c->lat_n2 = c->lat_n3 = 0;
  } else {
    if (na < 1 || n1 < 1 || n2 < 1 || n3 < 1 || (int64_t)na * n1 * n2 * n3 != c->N)
      return fail(UASD_ERR_ARG, "NA*N1*N2*N3 must equal natom");
    c->lat_na = na;
    c->lat_n1 = n1;
    c->lat_n2 = n2;
    c->lat_n3 = n3;
  }
  c->stencil_dirty = true;
  c->tile_off_shape = 0;
  c->gen += 1;
  return UASD_OK;
}

int uasd_has_stencil(uasd_ctx *c, int *has, int *radius) {
  if (int r = check_ctx(c)) return r;
  build_stencil(c);
  if (has) *has = c->stencil_ok ? 1 : 0;
  if (radius) {
    radius[0] = std::max(c->st_ex.rx, c->st_dm.rx);
    radius[1] = std::max(c->st_ex.ry, c->st_dm.ry);
    radius[2] = std::max(c->st_ex.rz, c->st_dm.rz);
  }
  return UASD_OK;
}

int uasd_set_segments(uasd_ctx *c, int nseg, const int *offsets) {
  if (int r = check_ctx(c)) return r;
  if (nseg > 1 && c->order_na > 1)
    return fail(UASD_ERR_UNSUPPORTED, "segments need the reference site order");
  if (nseg <= 0 || !offsets) return fail(UASD_ERR_ARG, "nseg must be > 0 with offsets (nseg+1)");
  if (offsets[0] != 0 || offsets[nseg] != c->N)
    return fail(UASD_ERR_ARG, "segment offsets must start at 0 and end at natom");
  for (int s = 0; s < nseg; ++s)
    if (offsets[s + 1] <= offsets[s]) return fail(UASD_ERR_ARG, "segments must be non-empty and increasing");
  return set_segments(c, nseg, offsets);
}

int uasd_measure_segments(uasd_ctx *c, double *msum, double *energy) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_state) return fail(UASD_ERR_STATE, "moments not set");
  if (!msum) return fail(UASD_ERR_ARG, "msum is null");
  if (int r = ensure_segments(c)) return r;
  if (energy) {
    if (!c->have_ex) return fail(UASD_ERR_STATE, "exchange not set");
    if (int r = rebuild_classes(c)) return r;
    int r = c->prec == UASD_FP64 ? run_field<double>(c, false, true, false, false)
                                 : run_field<float>(c, false, true, false, false);
    if (r) return r;
  }
  int r = c->prec == UASD_FP64 ? segment_sums<double>(c, energy != nullptr)
                               : segment_sums<float>(c, energy != nullptr);
  if (r) return r;
  const int nv = energy ? 4 : 3;
  std::vector<double> out((size_t)c->nseg * c->M * nv);
  HIP_TRY(hipMemcpyAsync(out.data(), c->seg_out.p, out.size() * sizeof(double),
                         hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  for (size_t t = 0; t < (size_t)c->nseg * c->M; ++t) {
    for (int d = 0; d < 3; ++d) msum[3 * t + d] = out[nv * t + d];
    if (energy) energy[t] = out[nv * t + 3] * uasd::kMub / uasd::kMry;
  }
  return UASD_OK;
}

}  // extern "C"

namespace {

// calc_energy's four terms per (segment, ensemble) into ene (4,M,nseg), with
// the chunk partials in `partial` (nchunks*M*4 doubles) and the sums in `sums`
// (nseg*M*4 doubles), both device memory.  The sums are copied straight into
// ene and scaled there, so no host memory is taken either.
int energy_terms_into(uasd_ctx *c, double *partial, double *sums, double *ene) {
  const int2 *chunks = c->seg_dev.as<int2>();
  const int *seg_chunk = reinterpret_cast<const int *>(chunks + c->nchunks);
  if (c->prec == UASD_FP64) {
    HIP_TRY(uasd::launch_energy_terms<double>(c->stream, ham_view<double>(c), c->nseg,
                                              c->nchunks, chunks, seg_chunk,
                                              quads<double>(c, c->spins, 0), partial, sums));
  } else {
    HIP_TRY(uasd::launch_energy_terms<float>(c->stream, ham_view<float>(c), c->nseg,
                                             c->nchunks, chunks, seg_chunk,
                                             quads<float>(c, c->spins, 0), partial, sums));
  }
  const size_t n = (size_t)c->nseg * c->M * 4;
  HIP_TRY(hipMemcpyAsync(ene, sums, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  // per site in mRy: energy.f90:353-366 divides by the number of atoms,
  // calculate_mean_and_deviation then scales by mub/mry
  for (int sg = 0; sg < c->nseg; ++sg) {
    const double na = (double)(c->seg_off[sg + 1] - c->seg_off[sg]);
    for (int k = 0; k < c->M; ++k)
      for (int t = 0; t < 4; ++t) {
        const size_t i = ((size_t)sg * c->M + k) * 4 + t;
        ene[i] = ene[i] / na * (uasd::kMub / uasd::kMry);
      }
  }
  return UASD_OK;
}

int energy_terms_check(uasd_ctx *c, double *ene) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_state) return fail(UASD_ERR_STATE, "moments not set");
  if (!c->have_ex) return fail(UASD_ERR_STATE, "exchange not set");
  if (!ene) return fail(UASD_ERR_ARG, "ene is null");
  if (c->M > 65535) return fail(UASD_ERR_UNSUPPORTED, "more than 65535 ensembles");
  return UASD_OK;
}

}  // namespace

extern "C" {

int uasd_energy_terms(uasd_ctx *c, double *ene) {
  if (int r = energy_terms_check(c, ene)) return r;
  if (int r = ensure_segments(c)) return r;
  if (int r = rebuild_classes(c)) return r;
  HIP_TRY(c->seg_partial.ensure((size_t)c->nchunks * c->M * 4 * sizeof(double)));
  HIP_TRY(c->seg_out.ensure((size_t)c->nseg * c->M * 4 * sizeof(double)));
  return energy_terms_into(c, c->seg_partial.as<double>(), c->seg_out.as<double>(), ene);
}

int uasd_energy_terms_noalloc(uasd_ctx *c, double *ene) {
  if (int r = energy_terms_check(c, ene)) return r;
  if (c->nseg == 0) return fail(UASD_ERR_STATE, "the context has no segments");
  const size_t need = ((size_t)c->nchunks + (size_t)c->nseg) * (size_t)c->M * 4;
  if (need > kScratchDoubles)
    return fail(UASD_ERR_ARG,
                "uasd_energy_terms_noalloc needs " + std::to_string(need) +
                    " doubles of scratch, more than its fixed " + std::to_string(kScratchDoubles) +
                    ": (chunks of up to 4096 sites + segments) * ensembles * 4 must not exceed it; "
                    "use uasd_energy_terms");
  double *base = scratch_of(c->device);
  if (!base) return fail(UASD_ERR_STATE, "no scratch address for this device");
  if (int r = rebuild_classes(c, false)) return r;
  return energy_terms_into(c, base, base + (size_t)c->nchunks * c->M * 4, ene);
}

int uasd_accumulate(uasd_ctx *c, int with_energy) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_state) return fail(UASD_ERR_STATE, "moments not set");
  if (int r = ensure_segments(c)) return r;
  if (with_energy) {
    if (!c->have_ex) return fail(UASD_ERR_STATE, "exchange not set");
    if (int r = rebuild_classes(c)) return r;
    int r = c->prec == UASD_FP64 ? run_field<double>(c, false, true, false, false)
                                 : run_field<float>(c, false, true, false, false);
    if (r) return r;
  }
  int r = c->prec == UASD_FP64 ? segment_sums<double>(c, with_energy != 0)
                               : segment_sums<float>(c, with_energy != 0);
  if (r) return r;
  const int *seg_n = reinterpret_cast<const int *>(c->seg_dev.as<int2>() + c->nchunks) + c->nseg + 1;
  HIP_TRY(uasd::launch_accumulate(c->stream, c->nseg, c->M, seg_n, c->seg_out.as<double>(),
                                  with_energy ? 4 : 3, c->acc.as<double>()));
  c->acc_samples += 1;
  return UASD_OK;
}

int uasd_get_accumulators(uasd_ctx *c, double *out, int64_t *nsamples) {
  if (int r = check_ctx(c)) return r;
  if (int r = ensure_segments(c)) return r;
  if (out) {
    HIP_TRY(hipMemcpyAsync(out, c->acc.p, (size_t)c->nseg * c->M * uasd::kAccWidth * sizeof(double),
                           hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
  }
  if (nsamples) *nsamples = c->acc_samples;
  return UASD_OK;
}

int uasd_reset_accumulators(uasd_ctx *c) {
  if (int r = check_ctx(c)) return r;
  if (c->nseg == 0) return ensure_segments(c);
  std::vector<int> off(c->seg_off);
  return set_segments(c, c->nseg, off.data());
}

int uasd_get_coloring(uasd_ctx *c, int *ncolors, int *color_of_site) {
  if (int r = check_ctx(c)) return r;
  if (!c->have_ex) return fail(UASD_ERR_STATE, "exchange not set");
  if (int r = build_coloring(c)) return r;
  if (ncolors) *ncolors = c->ncolors;
  if (color_of_site)
    for (int i = 0; i < c->N; ++i) color_of_site[i] = c->color_of_site[slot_of(c, i)];
  return UASD_OK;
}

int uasd_set_kernel_timing(uasd_ctx *c, int enable) {
  if (int r = check_ctx(c)) return r;
  if (int r = resolve_timing(c)) return r;
  if (enable < -1) return fail(UASD_ERR_ARG, "enable must be >= -1");
  c->timing = enable > 0;
  c->timing_every = enable > 0 ? enable : 1;
  c->timing_region = enable != 0;
  for (auto &t : c->timers) t = Timing{};
  for (auto &k : c->timing_tick) k = 0;
  return UASD_OK;
}

int uasd_get_kernel_timing(uasd_ctx *c, int kind, int64_t *launches, double *total_ms) {
  if (int r = check_ctx(c)) return r;
  if (kind < 0 || kind > 6) return fail(UASD_ERR_ARG, "kind must be 0..6");
  if (int r = resolve_timing(c)) return r;
  if (launches) *launches = c->timers[kind].launches;
  if (total_ms) *total_ms = c->timers[kind].ms;
  return UASD_OK;
}

}  // extern "C"
