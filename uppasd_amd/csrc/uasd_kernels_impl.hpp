// uasd_kernels_impl.hpp -- definitions of the launchers declared in
// uasd_launch.hpp, instantiated for one arithmetic type by the including
// translation unit.
#pragma once
#include <algorithm>
#include <type_traits>

#include "uasd_launch.hpp"

namespace uasd {

// Calls f(std::integral_constant<int, G>) for the gather width of t.
template <typename F>
static hipError_t with_gather(const Tune &t, F &&f) {
  switch (t.gather) {
    case 2: return f(std::integral_constant<int, 2>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 8: return f(std::integral_constant<int, 8>{});
    case 16: return f(std::integral_constant<int, 16>{});
    default: return hipErrorInvalidValue;
  }
}

template <typename R>
hipError_t launch_field(hipStream_t s, const Tune &t, const HamDev<R> &h, const Quad<R> *src,
                        Quad<R> *beff, double *en, Quad<R> *parts) {
  const int64_t n = (int64_t)h.N * h.M;
  if (n == 0) return hipSuccess;
  if (!tune_valid(t)) return hipErrorInvalidValue;
  const HamDev<R> hh = tuned(h, t);
  return with_gather(t, [&](auto g) {
    hipLaunchKernelGGL((k_field<R, decltype(g)::value>), dim3(grid_for(n, t.block)),
                       dim3(t.block), 0, s, hh, src, beff, en, parts);
    return hipGetLastError();
  });
}

template <typename R, int ALG, int HALF, bool FUSED>
static hipError_t llg_one(Queue s, const Tune &t, const HamDev<R> &h,
                          const LLGDev<R> &prm, const Quad<R> *e, Quad<R> *p, Quad<R> *b2,
                          const Quad<R> *beff, Quad<R> *out) {
  const int64_t n = (int64_t)h.N * h.M;
  if (n == 0) return hipSuccess;
  const dim3 grid(grid_for(n, t.block)), block(t.block);
  const HamDev<R> hh = tuned(h, t);
  if (!FUSED) {  // no gather: one instance
    return enqueue(s, k_llg<R, ALG, HALF, false, 4>, grid, block, 0, hh, prm, e, p, b2, beff, out);
  }
  return with_gather(t, [&](auto g) {
    return enqueue(s, k_llg<R, ALG, HALF, true, decltype(g)::value>, grid, block, 0, hh, prm, e, p,
                   b2, beff, out);
  });
}

template <typename R>
hipError_t launch_llg(Queue s, const Tune &t, int alg, int half, bool fused,
                      const HamDev<R> &h, const LLGDev<R> &prm, const Quad<R> *e, Quad<R> *p,
                      Quad<R> *b2, const Quad<R> *beff, Quad<R> *out) {
  if (!tune_valid(t)) return hipErrorInvalidValue;
#define UASD_LLG_CASE(A, H, F)             \
  if (alg == A && half == H && fused == F) \
    return llg_one<R, A, H, F>(s, t, h, prm, e, p, b2, beff, out);
  UASD_LLG_CASE(1, 0, true)
  UASD_LLG_CASE(1, 1, true)
  UASD_LLG_CASE(1, 0, false)
  UASD_LLG_CASE(1, 1, false)
  UASD_LLG_CASE(4, 0, true)
  UASD_LLG_CASE(4, 1, true)
  UASD_LLG_CASE(4, 0, false)
  UASD_LLG_CASE(4, 1, false)
  UASD_LLG_CASE(6, 0, true)
  UASD_LLG_CASE(6, 1, true)
  UASD_LLG_CASE(6, 0, false)
  UASD_LLG_CASE(6, 1, false)
  UASD_LLG_CASE(7, 0, true)
  UASD_LLG_CASE(7, 1, true)
  UASD_LLG_CASE(7, 0, false)
  UASD_LLG_CASE(7, 1, false)
  UASD_LLG_CASE(5, 0, true)
  UASD_LLG_CASE(5, 1, true)
  UASD_LLG_CASE(5, 0, false)
  UASD_LLG_CASE(5, 1, false)
#undef UASD_LLG_CASE
  return hipErrorInvalidValue;
}

template <typename R>
hipError_t launch_draw(Queue s, const HamDev<R> &h, const LLGDev<R> &prm, int steps,
                       Quad<R> *out) {
  const int64_t n = (int64_t)h.N * h.M;
  if (n == 0 || steps <= 0) return hipSuccess;
  const int block = n <= 64 * 256 ? 64 : kBlock;
  return enqueue(s, k_draw<R>, dim3((unsigned)((n + block - 1) / block), (unsigned)steps),
                 dim3(block), 0, h, prm, steps, out);
}

template <typename R>
hipError_t launch_mc(Queue s, const Tune &t, const HamDev<R> &h, const MCParams &mp,
                     Quad<R> *spins) {
  const int64_t n = (int64_t)mp.nsites * h.M;
  if (n == 0) return hipSuccess;
  if (!tune_valid(t)) return hipErrorInvalidValue;
  const HamDev<R> hh = tuned(h, t);
  // two adjacent ensembles per thread where M is even
  const bool two = t.pair && h.M % 2 == 0;
  MCParams m = mp;
  m.pdiv = make_fast_div((uint32_t)(two ? h.M / 2 : h.M));
  return with_gather(t, [&](auto g) {
    constexpr int G = decltype(g)::value;
    const dim3 grid(grid_for(two ? n / 2 : n, t.block)), block(t.block);
    if (mp.heat_bath)
      return two ? enqueue(s, k_mc_colour<R, G, 2, true>, grid, block, 0, hh, m, spins)
                 : enqueue(s, k_mc_colour<R, G, 1, true>, grid, block, 0, hh, m, spins);
    return two ? enqueue(s, k_mc_colour<R, G, 2, false>, grid, block, 0, hh, m, spins)
               : enqueue(s, k_mc_colour<R, G, 1, false>, grid, block, 0, hh, m, spins);
  });
}

template <typename R, int ALG, bool LNB>
static hipError_t llg_resident_one(hipStream_t s, const HamDev<R> &h, const LLGDev<R> &prm,
                                   const ResDev &rd, int nsteps, size_t bytes, int threads,
                                   Quad<R> *spins) {
  static LdsLimit limit;
  const hipError_t err = limit.raise((const void *)&k_llg_resident<R, ALG, LNB>, bytes);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL((k_llg_resident<R, ALG, LNB>), dim3((unsigned)(rd.ncomp * h.M)),
                     dim3(threads), bytes, s, h, prm, rd, nsteps, spins);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_llg_resident(hipStream_t s, int alg, const HamDev<R> &h, const LLGDev<R> &prm,
                               const ResDev &rd, int nsteps, size_t lds, Quad<R> *spins) {
  const size_t base = res_lds_llg(sizeof(R), rd.nmax), lists = 2 * (size_t)rd.nmax * (h.W + h.Wd);
  if (base > lds || nsteps <= 0) return hipErrorInvalidValue;
  const int threads = std::min(kResThreads, (rd.nmax + 63) / 64 * 64);
  const bool lnb = res_lists_in_lds((int64_t)rd.ncomp * h.M, threads, 16, base, lists, lds);
  const size_t bytes = base + (lnb ? lists : 0);
#define UASD_RES_CASE(A)                                                                       \
  if (alg == A)                                                                                \
    return lnb ? llg_resident_one<R, A, true>(s, h, prm, rd, nsteps, bytes, threads, spins)    \
               : llg_resident_one<R, A, false>(s, h, prm, rd, nsteps, bytes, threads, spins);
  UASD_RES_CASE(1)
  UASD_RES_CASE(4)
  UASD_RES_CASE(5)
  UASD_RES_CASE(6)
  UASD_RES_CASE(7)
#undef UASD_RES_CASE
  return hipErrorInvalidValue;
}

template <typename R, bool HB, bool TRL, bool LNB>
static hipError_t mc_resident_one(Queue s, const HamDev<R> &h, const MCParams &mp,
                                  const ResDev &rd, int nsweeps, size_t bytes, int threads,
                                  Quad<R> *spins, Quad<R> *trials) {
  static LdsLimit limit;
  const hipError_t err = limit.raise((const void *)&k_mc_resident<R, HB, TRL, LNB>, bytes);
  if (err != hipSuccess) return err;
  return enqueue(s, k_mc_resident<R, HB, TRL, LNB>, dim3((unsigned)(rd.ncomp * h.M)),
                 dim3(threads), bytes, h, mp, rd, nsweeps, spins, trials);
}

template <typename R>
hipError_t launch_mc_resident(Queue s, const HamDev<R> &h, const MCParams &mp,
                              const ResDev &rd, int nsweeps, size_t lds, Quad<R> *spins,
                              Quad<R> *trials) {
  const size_t sp = res_lds_spins(sizeof(R), rd.nmax), lists = res_lds_lists(rd.nmax, h.W + h.Wd);
  const size_t tr = 4 * sizeof(R) * (size_t)rd.nmax;
  if (sp > lds || nsweeps <= 0) return hipErrorInvalidValue;
  // A phase needs a thread per site of its colour.  Only the trial moves of a
  // sweep can use more, and only while the chip has CUs to spare (256 of
  // them): with more systems than that the waves are better spent on other
  // workgroups (1024 heat-bath systems of 432 sites: 83 -> 30 us a sweep).
  const bool wide = !mp.heat_bath && (int64_t)rd.ncomp * h.M <= 512;
  const int threads = std::min(kResThreads, ((wide ? rd.nmax : rd.cmax) + 63) / 64 * 64);
  // the trials of a sweep in LDS where they fit, then the lists
  const bool trl = !mp.heat_bath && sp + tr <= lds;
  const size_t base = sp + (trl ? tr : 0);
  const int cu_waves = sizeof(R) == 8 && !mp.heat_bath ? 8 : 16;
  const bool lnb = res_lists_in_lds((int64_t)rd.ncomp * h.M, threads, cu_waves, base, lists, lds);
  const size_t bytes = base - 16 + (lnb ? lists : 0);  // the counters are static
#define UASD_RES_CASE(HB_, TRL_, LNB_)                                                          \
  if ((mp.heat_bath != 0) == HB_ && trl == TRL_ && lnb == LNB_)                                 \
    return mc_resident_one<R, HB_, TRL_, LNB_>(s, h, mp, rd, nsweeps, bytes, threads, spins,    \
                                               trials);
  UASD_RES_CASE(true, false, true)
  UASD_RES_CASE(true, false, false)
  UASD_RES_CASE(false, true, true)
  UASD_RES_CASE(false, true, false)
  UASD_RES_CASE(false, false, true)
  UASD_RES_CASE(false, false, false)
#undef UASD_RES_CASE
  return hipErrorInvalidValue;
}

template <typename R>
hipError_t launch_llg_tile(Queue s, TileDev t, int pipe, int alg, int half,
                           const HamDev<R> &h, const LLGDev<R> &prm, const Quad<R> *e,
                           Quad<R> *p, Quad<R> *b2, Quad<R> *out) {
  switch (alg) {
    case 1: return launch_llg_tile_alg<R, 1>(s, t, pipe, half, h, prm, e, p, b2, out);
    case 4: return launch_llg_tile_alg<R, 4>(s, t, pipe, half, h, prm, e, p, b2, out);
    case 5: return launch_llg_tile_alg<R, 5>(s, t, pipe, half, h, prm, e, p, b2, out);
    case 6: return launch_llg_tile_alg<R, 6>(s, t, pipe, half, h, prm, e, p, b2, out);
    case 7: return launch_llg_tile_alg<R, 7>(s, t, pipe, half, h, prm, e, p, b2, out);
    default: return hipErrorInvalidValue;
  }
}

template <typename R>
hipError_t launch_reduce(hipStream_t s, int N, int M, const Quad<R> *spins, const double *en,
                         int nv, double *partial, int nblocks, double *out) {
  if (N == 0 || M == 0) return hipSuccess;
  const int chunk = (N + nblocks - 1) / nblocks;
  dim3 g1(nblocks, M);
  if (nv == 4) {
    hipLaunchKernelGGL((k_reduce_stage1<R, 4>), g1, dim3(kBlock), 0, s, N, M, chunk, spins, en,
                       partial);
    hipLaunchKernelGGL(k_reduce_stage2<4>, dim3(M), dim3(kBlock), 0, s, M, nblocks,
                       partial, out);
  } else {
    hipLaunchKernelGGL((k_reduce_stage1<R, 3>), g1, dim3(kBlock), 0, s, N, M, chunk, spins, en,
                       partial);
    hipLaunchKernelGGL(k_reduce_stage2<3>, dim3((M * 3 + 3) / 4), dim3(kBlock), 0, s, M, nblocks,
                       partial, out);
  }
  return hipGetLastError();
}

// The chunk partials of every (segment, ensemble, value) summed.
template <int NV>
static hipError_t segsum_final(hipStream_t s, int nseg, int M, int nchunks, const int *seg_chunk,
                               const double *partial, double *out) {
  const bool wave = nchunks >= 16 * (int64_t)nseg;  // many chunks per segment
  const int64_t per = wave ? 4 : 32, n = (int64_t)nseg * M * NV;  // sums per workgroup
  const dim3 grid((unsigned)std::min<int64_t>((n + per - 1) / per, 1 << 16));
  if (wave)
    hipLaunchKernelGGL((k_segsum_final<NV, 64>), grid, dim3(kBlock), 0, s, nseg, M, seg_chunk,
                       partial, out);
  else
    hipLaunchKernelGGL((k_segsum_final<NV, 8>), grid, dim3(kBlock), 0, s, nseg, M, seg_chunk,
                       partial, out);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_segsum(hipStream_t s, int M, int nseg, int nchunks, const int2 *chunks,
                         const int *seg_chunk, const Quad<R> *spins, const double *en, int nv,
                         double *partial, double *out) {
  if (nseg == 0 || M == 0 || nchunks == 0) return hipSuccess;
  const bool wide = kBlock % M == 0;
  const dim3 g = wide ? dim3(nchunks) : dim3(nchunks, M);
  if (nv == 4) {
    if (wide)
      hipLaunchKernelGGL((k_segsum_wide<R, 4>), g, dim3(kBlock), 0, s, M, chunks, spins, en,
                         partial);
    else
      hipLaunchKernelGGL((k_segsum_strided<R, 4>), g, dim3(kBlock), 0, s, M, chunks, spins, en,
                         partial);
    return segsum_final<4>(s, nseg, M, nchunks, seg_chunk, partial, out);
  }
  if (wide)
    hipLaunchKernelGGL((k_segsum_wide<R, 3>), g, dim3(kBlock), 0, s, M, chunks, spins, en, partial);
  else
    hipLaunchKernelGGL((k_segsum_strided<R, 3>), g, dim3(kBlock), 0, s, M, chunks, spins, en,
                       partial);
  return segsum_final<3>(s, nseg, M, nchunks, seg_chunk, partial, out);
}

template <typename R>
hipError_t launch_energy_terms(hipStream_t s, const HamDev<R> &h, int nseg, int nchunks,
                               const int2 *chunks, const int *seg_chunk, const Quad<R> *spins,
                               double *partial, double *out) {
  if (nseg == 0 || h.M == 0 || nchunks == 0) return hipSuccess;
  hipLaunchKernelGGL((k_energy_terms<R>), dim3(nchunks, h.M), dim3(kBlock), 0, s, h, chunks,
                     spins, partial);
  return segsum_final<4>(s, nseg, h.M, nchunks, seg_chunk, partial, out);
}

#define UASD_INSTANTIATE(R)                                                                   \
  template hipError_t launch_field<R>(hipStream_t, const Tune &, const HamDev<R> &,           \
                                      const Quad<R> *, Quad<R> *, double *, Quad<R> *);       \
  template hipError_t launch_llg<R>(Queue, const Tune &, int, int, bool,                \
                                    const HamDev<R> &, const LLGDev<R> &, const Quad<R> *,    \
                                    Quad<R> *, Quad<R> *, const Quad<R> *, Quad<R> *);        \
  template hipError_t launch_draw<R>(Queue, const HamDev<R> &, const LLGDev<R> &, int,   \
                                     Quad<R> *);                                              \
  template hipError_t launch_mc<R>(Queue, const Tune &, const HamDev<R> &,              \
                                   const MCParams &, Quad<R> *);                              \
  template hipError_t launch_llg_resident<R>(hipStream_t, int, const HamDev<R> &,             \
                                             const LLGDev<R> &, const ResDev &, int, size_t,  \
                                             Quad<R> *);                                      \
  template hipError_t launch_mc_resident<R>(Queue, const HamDev<R> &, const MCParams &,  \
                                            const ResDev &, int, size_t, Quad<R> *, Quad<R> *); \
  template hipError_t launch_llg_tile<R>(Queue, TileDev, int, int, int,              \
                                         const HamDev<R> &, const LLGDev<R> &,                \
                                         const Quad<R> *, Quad<R> *, Quad<R> *, Quad<R> *);   \
  template hipError_t launch_reduce<R>(hipStream_t, int, int, const Quad<R> *, const double *, \
                                       int, double *, int, double *);                         \
  template hipError_t launch_segsum<R>(hipStream_t, int, int, int, const int2 *, const int *,  \
                                       const Quad<R> *, const double *, int, double *,        \
                                       double *);                                             \
  template hipError_t launch_energy_terms<R>(hipStream_t, const HamDev<R> &, int, int,        \
                                             const int2 *, const int *, const Quad<R> *,      \
                                             double *, double *);

}  // namespace uasd
