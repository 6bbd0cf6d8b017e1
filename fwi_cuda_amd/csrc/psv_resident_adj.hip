// psv_resident_adj.hip -- the resident propagation's adjoint kernels (psv_resident.h).
#include "psv_resident.h"

namespace psv {

hipError_t launch_resident_adjoint(const ResArgs<float> &r, const ResPlan &p, int N, int shots, hipStream_t st) {
    return launch_resident_t<float, true>(r, N, p.cpt, shots * p.ntx * p.ntz, p.threads, p.lds, st);
}

}  // namespace psv
