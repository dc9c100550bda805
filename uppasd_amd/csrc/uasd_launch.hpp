// uasd_launch.hpp -- host-callable launchers for the kernels in
// uasd_kernels.hpp.  Each arithmetic type is instantiated in its own
// translation unit (uasd_kernels_f64.hip / uasd_kernels_f32.hip) so the FP64
// unit can be compiled without multiply-add contraction.
#pragma once
#include <algorithm>
#include <map>
#include <mutex>

#include "uasd_kernels.hpp"

namespace uasd {

// Grid for n work items, padded to a multiple of the XCD count (the kernels
// remap blockIdx so each XCD takes a contiguous range; padding blocks exit).
inline unsigned grid_for(int64_t n, int block) {
  const int64_t b = (n + block - 1) / block;
  return (unsigned)((b + kXCD - 1) / kXCD * kXCD);
}

constexpr int kBlock = 256;  // largest workgroup the kernels are built for

// The dynamic LDS one kernel may be launched with (above 64 KiB it must be
// asked for).  That limit belongs to the process's kernel, which contexts on
// other threads launch too: it is only ever raised, one thread at a time, so
// no thread lowers it between another one's raise and launch.
struct LdsLimit {
  std::mutex mu;
  std::map<int, size_t> bytes;  // per device
  hipError_t raise(const void *kern, size_t n) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    std::lock_guard<std::mutex> lock(mu);
    size_t &have = bytes[dev];
    if (n <= have) return hipSuccess;
    err = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)n);
    if (err == hipSuccess) have = n;
    return err;
  }
};

// A graph under construction: its kernels run one after the other.
struct Recording {
  hipGraph_t graph = nullptr;
  hipGraphNode_t last = nullptr;
};

// Where a launch goes: to a stream, or to the end of a graph.  Graphs are built
// node by node, not captured from a stream: while any stream of the process is
// capturing, HIP refuses ordinary calls of other threads (hipDeviceSynchronize,
// legacy-stream copies), which in turn break the capture.
struct Queue {
  hipStream_t stream;
  Recording *rec = nullptr;
};

template <typename T>
struct Same {
  using type = T;
};

template <typename... P>
hipError_t enqueue(const Queue &q, void (*kern)(P...), dim3 grid, dim3 block, size_t lds,
                   typename Same<P>::type... args) {
  if (!q.rec) {
    hipLaunchKernelGGL(kern, grid, block, lds, q.stream, args...);
    return hipGetLastError();
  }
  void *params[] = {(void *)&args...};
  hipKernelNodeParams n{};
  n.func = (void *)kern;
  n.gridDim = grid;
  n.blockDim = block;
  n.sharedMemBytes = (unsigned)lds;
  n.kernelParams = params;  // copied by the call
  hipGraphNode_t node = nullptr;
  const hipError_t err =
      hipGraphAddKernelNode(&node, q.rec->graph, &q.rec->last, q.rec->last ? 1 : 0, &n);
  if (err == hipSuccess) q.rec->last = node;
  return err;
}

// Launch shape of the gathering kernels (chosen by the autotuner):
//   gather  neighbours whose loads are issued together: 2, 4, 8 or 16
//   block   workgroup size: 64, 128 or 256
//   nt      1: neighbour lists read with non-temporal loads
//   idx32   1: int32 list entries even where packed int16 entries exist
//   tile    fused LLG only: 0 = list gathers, k > 0 = LDS-tiled stencil with
//           tile shape kTileShapes[k-1] (periodic lattices with a stencil)
constexpr int kNumTileShapes = 15;
constexpr int kTileShapes[kNumTileShapes][3] = {
    {8, 8, 4}, {16, 8, 2}, {32, 4, 2}, {16, 4, 4}, {16, 16, 1}, {32, 8, 1}, {64, 4, 1}, {8, 4, 4},
    {4, 4, 4}, {8, 8, 2},  {16, 8, 1}, {8, 8, 1},  {16, 8, 4},  {8, 16, 4}, {8, 8, 8}};
struct Tune {
  int gather = 4;
  int block = 256;
  int nt = 0;
  int idx32 = 0;
  int tile = 0;
  int pipe = 0;  // tile kernel: 1 = resident workgroups loop over several tiles
  int pair = 0;  // MC colour pass: 1 = two adjacent ensembles per thread (M even)
  // 0: nobody has tuned, default_tune applies; kShapeAsked: set by the caller,
  // or the autotuner's fastest; kShapeResident: the autotuner's fastest shape,
  // for where resident launches, which were faster still, do not apply
  int chosen = 0;
};
constexpr int kShapeAsked = 1, kShapeResident = 2;

// Launch shape of a gathering kernel that nobody has tuned: n items (sites x
// ensembles of a launch), w neighbours.  A small launch is a chain of loads on
// a chip that is mostly idle: workgroups of one wavefront spread it over the
// most CUs and their caches, and with many neighbours eight gathers in flight
// halve the number of rounds.  LLG step at 58 neighbours, (4, 256) -> (8, 64):
// 16,000 sites FP64 24.4 -> 16.9 us, 65,536 sites 26.3 -> 24.2 us; 14
// neighbours -> (4, 64): 16,000 sites 13.5 -> 12.2 us, 65,536 sites equal.  MC
// sweep of 15,840 sites at 58 neighbours 338 -> 180 us.  From 2^18 items on
// the shapes are within a few per cent of each other.
inline Tune default_tune(const Tune &t, int64_t n, int w) {
  if (t.chosen || n > (int64_t)1 << 18) return t;
  Tune d = t;
  d.block = 64;
  d.gather = w >= 16 ? 8 : 4;
  return d;
}

inline bool tune_valid(const Tune &t) {
  return (t.gather == 2 || t.gather == 4 || t.gather == 8 || t.gather == 16) &&
         (t.block == 64 || t.block == 128 || t.block == 256) && (t.nt == 0 || t.nt == 1) &&
         (t.idx32 == 0 || t.idx32 == 1) && t.tile >= 0 && t.tile <= kNumTileShapes &&
         (t.pipe == 0 || (t.pipe == 1 && t.tile > 0)) &&
         (t.pair == 0 || (t.pair == 1 && t.tile == 0));
}

// The Hamiltonian view a launch uses under a tuning choice.
template <typename R>
inline HamDev<R> tuned(const HamDev<R> &h, const Tune &t) {
  HamDev<R> hh = h;
  hh.nt = t.nt;
  if (t.idx32) {
    hh.nbr16 = nullptr;
    hh.dnbr16 = nullptr;
  }
  return hh;
}

// parts (nullable) receives beff1 then beff2, N*M quads each.
template <typename R>
hipError_t launch_field(hipStream_t s, const Tune &t, const HamDev<R> &h, const Quad<R> *src,
                        Quad<R> *beff, double *en, Quad<R> *parts);

// alg: 1 midpoint / 5 Depondt; half: 0 predictor, 1 corrector
template <typename R>
hipError_t launch_llg(Queue s, const Tune &t, int alg, int half, bool fused,
                      const HamDev<R> &h, const LLGDev<R> &prm, const Quad<R> *e, Quad<R> *p,
                      Quad<R> *b2, const Quad<R> *beff, Quad<R> *out);

// Wavefronts that one phase of a system (a colour, a half step) of `sites`
// sites takes in a workgroup of `slots` wavefronts: at least one, and a quarter
// of the workgroup's, whose slots stay taken.
inline int res_waves(int sites, int slots) {
  return std::max({1, (sites + 63) / 64, slots / 4});
}

// Wavefronts of a phase (res_waves over all systems) less `weight` times the
// full ones that `items` sites would make: the idle share of a resident launch.
// A system takes a workgroup of at least one wavefront however few sites it
// has, so batches of many tiny systems are faster half step by half step or
// colour by colour; the callers' comments have the limits and their figures.
inline double res_idle_waves(int64_t waves, int64_t items, double weight) {
  return (double)waves - weight * (double)items / 64.0;
}

// Whether a resident launch keeps its lists in LDS beside `base` bytes of
// state: where they fit and do not make the workgroups take turns on a CU that
// would hold several at once without them (`lds` bytes and `cu_waves` wavefronts
// a CU, which the kernel's registers allow; 256 CUs).  1000 systems of 1024
// sites with 58 neighbours, lists of 119 KB in LDS (one workgroup a CU, four
// rounds) -> in global memory, us a sweep: FP32 Metropolis 327 -> 83, heat bath
// 370 -> 88, FP64 360 -> 86 (colour by colour 180, 186, 283); 260 systems
// 97 -> 63, 186 -> 80, 169 -> 79.
inline bool res_lists_in_lds(int64_t systems, int threads, int cu_waves, size_t base,
                             size_t lists, size_t lds) {
  if (base + lists > lds) return false;
  auto rounds = [&](size_t bytes) {
    const int64_t cu =
        std::min<int64_t>(lds / std::max<size_t>(bytes, 1), std::max(1, 64 * cu_waves / threads));
    return (systems + 256 * cu - 1) / (256 * cu);
  };
  return rounds(base + lists) <= rounds(base);
}

// nsteps LLG steps of every system with k_llg_resident; Philox deviates in
// prm.nsave, lds = LDS bytes a workgroup may use.
template <typename R>
hipError_t launch_llg_resident(hipStream_t s, int alg, const HamDev<R> &h, const LLGDev<R> &prm,
                               const ResDev &rd, int nsteps, size_t lds, Quad<R> *spins);

// LDS of k_llg_resident without its lists: e, p and b2 quads.
inline size_t res_lds_llg(size_t rsize, int nmax) { return 12 * rsize * (size_t)nmax; }

// Deviates of `steps` steps from prm.step on into as many quad arrays of out.
template <typename R>
hipError_t launch_draw(Queue s, const HamDev<R> &h, const LLGDev<R> &prm, int steps,
                       Quad<R> *out);

template <typename R>
hipError_t launch_mc(Queue s, const Tune &t, const HamDev<R> &h, const MCParams &mp,
                     Quad<R> *spins);

// nsweeps sweeps of every system with k_mc_resident; lds = LDS bytes a
// workgroup may use, trials = N*M quads of scratch for the trial moves that do
// not fit in them (not read before they are written).
template <typename R>
hipError_t launch_mc_resident(Queue s, const HamDev<R> &h, const MCParams &mp,
                              const ResDev &rd, int nsweeps, size_t lds, Quad<R> *spins,
                              Quad<R> *trials);

// LDS of k_mc_resident with nmax sites: what it cannot do without (the spins,
// the sorted positions and two counters), and w list entries per site.
inline size_t res_lds_lists(int nmax, int w) { return sizeof(uint16_t) * (size_t)nmax * w; }
inline size_t res_lds_spins(size_t rsize, int nmax) {
  return 4 * rsize * (size_t)nmax + res_lds_lists(nmax, rsize == 8 ? 1 : 0) + 16;
}

// Fused LLG half-step with the LDS-tiled stencil kernel, work units (tile,
// ensemble).
template <typename R>
hipError_t launch_llg_tile(Queue s, TileDev t, int pipe, int alg, int half,
                           const HamDev<R> &h, const LLGDev<R> &prm, const Quad<R> *e,
                           Quad<R> *p, Quad<R> *b2, Quad<R> *out);
// The same for one solver; uasd_tile.hip instantiates each (R, ALG).
template <typename R, int ALG>
hipError_t launch_llg_tile_alg(Queue s, TileDev t, int pipe, int half, const HamDev<R> &h,
                               const LLGDev<R> &prm, const Quad<R> *e, Quad<R> *p, Quad<R> *b2,
                               Quad<R> *out);
// LDS bytes the tile kernel needs for a halo tile of hv cells
// Component plane size of k_llg_tile for NA*HV halo values: the smallest of
// kTilePlanes that holds them, or 0.
inline int tile_plane(int nahv) {
  for (int k = 0; k < kNumTilePlanes; ++k)
    if (nahv <= kTilePlanes[k]) return kTilePlanes[k];
  return 0;
}
// LDS of k_llg_tile: three planes of `plane` values (NA*HV used), then two
// staging tables of the halo (ntab = HX + NA*HY*HZ ints each)
inline size_t tile_lds_bytes(size_t rsize, int plane, int ntab) {
  return 3 * (size_t)plane * rsize + 2 * (size_t)ntab * sizeof(int);
}

// FP64 sums per ensemble of emomM (nv = 3) or of emomM and en (nv = 4);
// partial must hold M*nblocks*nv doubles, out M*nv doubles.
template <typename R>
hipError_t launch_reduce(hipStream_t s, int N, int M, const Quad<R> *spins, const double *en,
                         int nv, double *partial, int nblocks, double *out);

// Per-segment FP64 sums (see k_segsum_*): chunks (nchunks), seg_chunk
// (nseg+1, chunk ranges of each segment), partial (nchunks*M*nv doubles),
// out (nseg*M*nv doubles).
template <typename R>
hipError_t launch_segsum(hipStream_t s, int M, int nseg, int nchunks, const int2 *chunks,
                         const int *seg_chunk, const Quad<R> *spins, const double *en, int nv,
                         double *partial, double *out);

// Term-resolved energies (see k_energy_terms) per (segment, ensemble):
// out[(seg*M + ens)*4 + t] for t = exchange, anisotropy, DM, Zeeman, sums
// over the segment's sites in field units; partial holds nchunks*M*4 doubles.
template <typename R>
hipError_t launch_energy_terms(hipStream_t s, const HamDev<R> &h, int nseg, int nchunks,
                               const int2 *chunks, const int *seg_chunk, const Quad<R> *spins,
                               double *partial, double *out);

// ctr[idx] = value (add = 0) or ctr[idx] += value (add = 1), on the stream.
hipError_t launch_counter(Queue s, int idx, uint64_t *ctr, uint64_t value, int add);

// Appends one cumulant sample per (segment, ensemble) from out of launch_segsum.
hipError_t launch_accumulate(hipStream_t s, int nseg, int M, const int *seg_n,
                             const double *sums, int nv, double *acc);

}  // namespace uasd
