// psv_resident_f64.hip -- the resident propagation in FP64, for seis_fp64 (psv_resident.h).
#include "psv_resident.h"

namespace psv {

hipError_t launch_resident_fp64(const ResArgs<double> &r, const ResPlan &p, int N, int shots, hipStream_t st) {
    return launch_resident_t<double, false>(r, N, p.cpt, shots * p.ntx * p.ntz, p.threads, p.lds, st);
}

}  // namespace psv
