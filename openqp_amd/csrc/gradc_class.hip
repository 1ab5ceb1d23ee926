// gradc_class.hip -- instantiates the cooperative gradient kernel of one quartet
// class (XA XB | XC XD).  Built once per class with -DXA=.. -DXB=.. -DXC=.. -DXD=..
#include "gradc_device.h"

namespace oqph {

#define OQPH_GRC_NAME_(p, a, b, c, d) p##a##b##c##d
#define OQPH_GRC_NAME(p, a, b, c, d) OQPH_GRC_NAME_(p, a, b, c, d)

static_assert(GRC<XA, XB, XC, XD>::fits, "the class does not fit the cooperative gradient kernel");

void OQPH_GRC_NAME(launch_gradc_, XA, XB, XC, XD)(const GradParams& p, const WaveWork& ww, hipStream_t s) {
  const int kpb = ww.kpb > 0 ? ww.kpb : 64;
  hipLaunchKernelGGL((k_gradc<XA, XB, XC, XD>), dim3((unsigned)(ww.nwaves * (64 / kpb))), dim3(64),
                     sizeof(double) * 3 * p.natm, s, p, ww);
}

bool OQPH_GRC_NAME(gradc_res_, XA, XB, XC, XD)(KernelRes* r) {
  hipFuncAttributes a;
  if (hipFuncGetAttributes(&a, (const void*)k_gradc<XA, XB, XC, XD>) != hipSuccess) return false;
  r->private_bytes = (int)a.localSizeBytes;
  r->lds_bytes = (int)a.sharedSizeBytes;
  r->regs = a.numRegs;
  r->max_threads = a.maxThreadsPerBlock;
  return true;
}

}  // namespace oqph
