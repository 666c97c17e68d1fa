// One-component-per-lane kernels (anchored binary32 RK4): the exact feature
// sets of the PIMM sweep, the R(H) loop and the VSD sweep, and the generic
// lean set (anisotropy, IEC, field drives of any kind); and the stochastic
// solvers (binary64 steps, binary32 normals) of the usual features.  Per step,
// against one lane per layer: 32 two-layer switching devices 0.52 -> 0.37 us,
// one-layer Euler-Heun devices at 300 K 1.13 -> 0.66, two-layer 0.89 -> 0.78,
// four-layer 1.05 -> 0.81.
#include "registry.h"
namespace cmtj {
static const KEntry kC[] = {
    CMTJ_KC(2, FM_PIMM, 1),  // the PIMM sweep: one Oersted step record
    CMTJ_KCLOG(2, FM_PIMM, 1),  // the same with its log layout compiled in
    CMTJ_KC(2, FM_PIMM, -1), CMTJ_KC(4, FM_PIMM, -1), CMTJ_KC(1, FM_RH, 0), CMTJ_KC(1, FM_VSD, 1),
    CMTJ_KCF(1, FM_VSD, 1), CMTJ_KCF(1, FM_LEAN, -1), CMTJ_KCF(2, FM_LEAN, -1), CMTJ_KCF(4, FM_LEAN, -1),
    CMTJ_KC(1, FM_LEAN, -1), CMTJ_KC(2, FM_LEAN, -1), CMTJ_KC(4, FM_LEAN, -1),
    CMTJ_KC32S(1, CMTJ_EULER_HEUN, FM_CIMS, 1), CMTJ_KC32S(2, CMTJ_EULER_HEUN, FM_CIMS, 1),
    CMTJ_KC32S(1, CMTJ_EULER_HEUN, FM_CPL, -1), CMTJ_KC32S(2, CMTJ_EULER_HEUN, FM_CPL, -1),
    CMTJ_KC32S(4, CMTJ_EULER_HEUN, FM_CPL, -1), CMTJ_KC32S(1, CMTJ_HEUN, FM_CPL, -1),
    CMTJ_KC32S(2, CMTJ_HEUN, FM_CPL, -1), CMTJ_KC32S(4, CMTJ_HEUN, FM_CPL, -1),
};
KTable kernels_cl() { return {kC, sizeof(kC) / sizeof(kC[0])}; }
}  // namespace cmtj
