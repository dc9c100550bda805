// Launcher of the LDS-tiled LLG kernels of one solver and one arithmetic type
// (UASD_ALG, UASD_REAL, given on the compiler's command line: each pair is a
// translation unit of its own, so the ten of them compile side by side).
#include "uasd_launch.hpp"

namespace uasd {

template <typename R, int ALG>
hipError_t launch_llg_tile_alg(Queue s, TileDev t, int pipe, int half, const HamDev<R> &h,
                               const LLGDev<R> &prm, const Quad<R> *e, Quad<R> *p, Quad<R> *b2,
                               Quad<R> *out) {
  // work units: (tile, ensemble) pairs
  const int64_t nunits64 = (int64_t)t.ntx * t.nty * t.ntz * h.M;
  if (nunits64 == 0) return hipSuccess;
  if (nunits64 >= (int64_t)1 << 31 || (int64_t)h.N * h.M >= (int64_t)1 << 31)
    return hipErrorInvalidValue;
  const int nunits = (int)nunits64;
  const int threads = t.TX * t.TY * t.TZ * t.NA;
  if (threads > 1024) return hipErrorInvalidValue;
  const int plane = tile_plane(t.NA * t.HV);
  // DM, anisotropy or Zeeman terms present: the full kernel
  const bool full = h.Wd > 0 || h.an_type != nullptr || h.ext_mode != 0;
  // several ensembles: the (tile, ensemble) unit instance
  const bool ens = h.M > 1;
  if (plane == 0) return hipErrorInvalidValue;
  if (t.rs < 1) return hipErrorInvalidValue;  // at least one halo row per round
  const size_t lds = tile_lds_bytes(sizeof(R), plane, t.HX + t.NA * t.HY * t.HZ);
  // one unit per workgroup, or (pipe) as many workgroups as are resident at
  // once (occupancy x CUs, kept per kernel for its last shape), each looping
  // over a run of consecutive units
  struct Slots {
    std::mutex mu;  // contexts on other threads launch the same kernel
    int dev = -1, threads = 0, n = 0;
    size_t lds = 0;
  };
  auto units_per_wg = [&](const void *kern, Slots &c) -> hipError_t {
    t.per = 1;
    if (!pipe) return hipSuccess;
    int dev = 0, ncu = 0, occ = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    std::lock_guard<std::mutex> lock(c.mu);
    if (c.dev != dev || c.lds != lds || c.threads != threads) {
      err = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
      if (err == hipSuccess)
        err = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, threads, lds);
      if (err != hipSuccess) return err;
      c.dev = dev;
      c.lds = lds;
      c.threads = threads;
      c.n = std::max(1, occ) * std::max(1, ncu);
    }
    t.per = (nunits + c.n - 1) / c.n;
    return hipSuccess;
  };
#define UASD_TILE_CASE(H, PL, F, E)                                                             \
  if (half == H && plane == PL && full == F && ens == E) {                                      \
    const auto kern = k_llg_tile<R, ALG, H, PL, F, E>;                                          \
    static LdsLimit limit;                                                                      \
    static Slots slots;                                                                         \
    hipError_t err = limit.raise((const void *)kern, lds);                                      \
    if (err == hipSuccess) err = units_per_wg((const void *)kern, slots);                       \
    if (err != hipSuccess) return err;                                                          \
    const int nwg = (nunits + t.per - 1) / t.per;                                               \
    const dim3 grid((nwg + kXCD - 1) / kXCD * kXCD), block(threads);                            \
    return enqueue(s, kern, grid, block, lds, tile_ham(h), prm, t, e, p, b2, out);              \
  }
#define UASD_TILE_FULL(H, PL)                                                                   \
  UASD_TILE_CASE(H, PL, false, false)                                                           \
  UASD_TILE_CASE(H, PL, true, false)                                                            \
  UASD_TILE_CASE(H, PL, false, true)                                                            \
  UASD_TILE_CASE(H, PL, true, true)
#define UASD_TILE_PLANES(H)                                                                     \
  UASD_TILE_FULL(H, kTilePlanes[0])                                                             \
  UASD_TILE_FULL(H, kTilePlanes[1])                                                             \
  UASD_TILE_FULL(H, kTilePlanes[2])                                                             \
  UASD_TILE_FULL(H, kTilePlanes[3])
  static_assert(kNumTilePlanes == 4, "one case per plane size");
  UASD_TILE_PLANES(0)
  UASD_TILE_PLANES(1)
#undef UASD_TILE_PLANES
#undef UASD_TILE_FULL
#undef UASD_TILE_CASE
  return hipErrorInvalidValue;
}

template hipError_t launch_llg_tile_alg<UASD_REAL, UASD_ALG>(Queue, TileDev, int, int,
                                                             const HamDev<UASD_REAL> &,
                                                             const LLGDev<UASD_REAL> &,
                                                             const Quad<UASD_REAL> *,
                                                             Quad<UASD_REAL> *, Quad<UASD_REAL> *,
                                                             Quad<UASD_REAL> *);

}  // namespace uasd
