// Dipole-coupled groups (Kanao and Nomura coupling) on one lane per vector
// component: the usual reservoir element (anisotropy, IEC, field drives) of
// one or two layers, binary64 RK4, 1 to 64 elements.
#include "registry.h"
namespace cmtj {
static const KEntry kGC[] = {
    CMTJ_KGC(1, FM_STATIC, 1), CMTJ_KGC(1, FM_STATIC, 2), CMTJ_KGC(1, FM_STATIC, 4),
    CMTJ_KGC(2, FM_STATIC, 1), CMTJ_KGC(2, FM_STATIC, 2), CMTJ_KGC(2, FM_STATIC, 4), CMTJ_KGC(2, FM_STATIC, 8),
    CMTJ_KGC(1, FM_LEAN, 1), CMTJ_KGC(1, FM_LEAN, 2), CMTJ_KGC(1, FM_LEAN, 4),
    CMTJ_KGC(2, FM_LEAN, 1), CMTJ_KGC(2, FM_LEAN, 2), CMTJ_KGC(2, FM_LEAN, 4), CMTJ_KGC(2, FM_LEAN, 8),
};
KTable kernels_group_cl() { return {kGC, sizeof(kGC) / sizeof(kGC[0])}; }
}  // namespace cmtj
