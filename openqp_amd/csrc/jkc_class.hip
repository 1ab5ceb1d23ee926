// jkc_class.hip -- instantiates the cooperative J/K kernel of one quartet
// class (XA XB | XC XD): Cartesian and pure AOs, closed- and open-shell pass.
// Built once per class with -DXA=.. -DXB=.. -DXC=.. -DXD=..
#include "jkc_device.h"
#include "launch_grid.h"

namespace oqph {

#define OQPH_JKC_NAME_(p, a, b, c, d) p##a##b##c##d
#define OQPH_JKC_NAME(p, a, b, c, d) OQPH_JKC_NAME_(p, a, b, c, d)

static_assert(jkc_fits<XA, XB, XC, XD>(), "the class does not fit the cooperative kernel");

template <bool PURE, bool TWO>
static void go(const JKParams& p, const WaveWork& ww, hipStream_t s) {
  const int kpb = ww.kpb > 0 ? ww.kpb : 64;
  const Grid2 g = wave_grid(ww.nwaves * (64 / kpb));
  hipLaunchKernelGGL((k_jkc<XA, XB, XC, XD, PURE, TWO>), dim3(g.x, g.y), dim3(64), 0, s, p, ww);
}

void OQPH_JKC_NAME(launch_jkc_, XA, XB, XC, XD)(bool pure, const JKParams& p, const WaveWork& ww, hipStream_t s) {
  if (p.F2) pure ? go<true, true>(p, ww, s) : go<false, true>(p, ww, s);
  else pure ? go<true, false>(p, ww, s) : go<false, false>(p, ww, s);
}

bool OQPH_JKC_NAME(jkc_res_, XA, XB, XC, XD)(bool pure, bool two, KernelRes* r) {
  const void* f = two ? (pure ? (const void*)k_jkc<XA, XB, XC, XD, true, true> : (const void*)k_jkc<XA, XB, XC, XD, false, true>)
                      : (pure ? (const void*)k_jkc<XA, XB, XC, XD, true, false> : (const void*)k_jkc<XA, XB, XC, XD, false, false>);
  hipFuncAttributes a;
  if (hipFuncGetAttributes(&a, f) != hipSuccess) return false;
  r->private_bytes = (int)a.localSizeBytes;
  r->lds_bytes = (int)a.sharedSizeBytes;
  r->regs = a.numRegs;
  r->max_threads = a.maxThreadsPerBlock;
  return true;
}

}  // namespace oqph
