// mpsa_svd.h -- host driver of the multi-workgroup sector SVD (mpsa_factor.hip),
// shared by the Chebyshev engine and the two-site split.
#pragma once
#include <algorithm>
#include <vector>

#include "mpsa_internal.h"

namespace mpsa {

// Chunk table of launch_house_panels / launch_house_apply: sector s has its
// workgroups at base[s] .. base[s + 1]; returns the largest min(m, n).
inline int house_table(const std::vector<SvdTask>& ts, int layout, std::vector<int>& base) {
  base.assign(ts.size() + 1, 0);
  int kmax = 0;
  for (size_t i = 0; i < ts.size(); ++i) {
    base[i + 1] = base[i] + house_chunks(ts[i].m, ts[i].n, layout);
    kmax = std::max(kmax, (int)std::min(ts[i].m, ts[i].n));
  }
  return kmax;
}

// The SVD of large sectors in phases: the load, the reflections in panels over
// several workgroups per sector, the init, sweeps of block-tournament rounds
// until a sweep rotates nothing (one host wait per sweep), the back-transform
// over several workgroups, the outputs (NaN where a sector does not converge).
// The blocks' order of pairs converges slowly where columns are many orders of
// magnitude apart (33 columns, half of them at 1e-60 of the others: 51 sweeps
// against 18 in the order of the one-workgroup kernel, at 1e-90 more than 60
// against 21), so that kernel finishes what still rotates after kSvdSweeps.
// Dev gives
//   const void* put(const std::vector<T>&)  a device copy ordered on the stream,
//                                           valid until the next wait after its use
//   void check(hipError_t, const char*)     throws on an error
//   void wait()                             drains the stream
// flags: big.size() doubles of device memory, zero.
template <class Dev>
void svd_blocked_run(Dev& dev, bool cplx, const std::vector<SvdTask>& big, const double* M, int64_t m_plane, double* U,
                     int64_t u_plane, double* Vt, int64_t vt_plane, double* S, double* W, int64_t w_plane,
                     double* flags, hipStream_t st) {
  const int nb = (int)big.size();
  std::vector<int> hbase;
  const int kmax = house_table(big, 0, hbase);
  const SvdTask* t = (const SvdTask*)dev.put(big);
  const int* dh = (const int*)dev.put(hbase);
  auto phase = [&](int ph, const char* what) {
    dev.check(launch_svd_phase(cplx, ph, t, nb, M, m_plane, U, u_plane, Vt, vt_plane, S, W, w_plane, st), what);
  };
  phase(kPhLoad, "sector SVD load");
  dev.check(launch_house_panels(cplx, 0, t, nb, dh, hbase.back(), kmax, W, w_plane, st), "sector SVD reflections");
  phase(kPhInit, "sector SVD init");
  // sweeps over the sectors still rotating: a sweep that rotates nothing in a
  // sector leaves it as it is, so later sweeps would not rotate it either
  std::vector<SvdTask> act = big;
  std::vector<double> hf((size_t)nb);
  for (int sweep = 0; sweep < kSvdSweeps && !act.empty(); ++sweep) {
    const int na = (int)act.size();
    std::vector<int> base((size_t)na + 1, 0);
    int rounds = 0, rmax = 1;
    for (int i = 0; i < na; ++i) {
      const SvdTask& a = act[(size_t)i];
      base[(size_t)i + 1] = base[(size_t)i] + svd_block_pairs(a.m, a.n);
      rounds = std::max(rounds, svd_block_rounds(a.m, a.n));
      rmax = std::max(rmax, (int)std::min(a.m, a.n));
    }
    const SvdTask* da = (const SvdTask*)dev.put(act);
    const int* db = (const int*)dev.put(base);
    for (int round = -1; round < rounds; ++round)
      dev.check(launch_svd_block_round(cplx, da, na, db, base.back(), round, W, w_plane, flags, rmax, st),
                "sector SVD round");
    dev.check(hipMemcpyAsync(hf.data(), flags, sizeof(double) * (size_t)na, hipMemcpyDeviceToHost, st),
              "sector SVD flags");
    dev.wait();
    std::vector<SvdTask> next;
    for (int i = 0; i < na; ++i)
      if (hf[(size_t)i] != 0.0) next.push_back(act[(size_t)i]);
    act.swap(next);
    if (!act.empty()) dev.check(launch_fill(flags, na, 0.0, st), "sector SVD flags");
  }
  if (!act.empty())
    dev.check(launch_svd_phase(cplx, kPhSweep, (const SvdTask*)dev.put(act), (int)act.size(), M, m_plane, U, u_plane,
                               Vt, vt_plane, S, W, w_plane, st),
              "sector SVD sweeps");
  phase(kPhBackInit, "sector SVD back-transform");
  dev.check(launch_house_apply(cplx, 0, t, nb, dh, hbase.back(), W, w_plane, st), "sector SVD back-transform");
  phase(kPhOut, "sector SVD outputs");
}

}  // namespace mpsa
